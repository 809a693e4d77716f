"""Storage in sweep-level order and the dataflow sweeps over it, at the shapes
where an order or a chunk can go wrong: one cell, levels of exactly 64 and of
65 cells, one-cell levels, a random numbering (many short levels), a colour
numbering (two to four levels of half the mesh), a batch.  Every comparison is
bitwise: the order only moves where a cell's data live."""
import numpy as np
import pytest

import phenlei_amd as pa

from conftest import perturbed_state

pytestmark = pytest.mark.gpu

FREE = np.array([1.0, 1.0, 0.0, 0.0, 1.0 / (1.4 * 0.25)])


def shapes():
    def shuffled():
        m = pa.Mesh.bump_hybrid(6, 3, 3, 1e-3, 4)
        return m.renumbered("perm", np.random.default_rng(3).permutation(m.n_cell))
    return {
        "one_cell": lambda: pa.Mesh.bump_hex(1, 1, 1),
        "line": lambda: pa.Mesh.bump_hex(9, 1, 1),
        "levels_of_64": lambda: pa.Mesh.bump_hex(64, 64, 1),
        "levels_of_65": lambda: pa.Mesh.bump_hex(65, 70, 1),
        "hybrid_shuffled": shuffled,
        "hex_coloured": lambda: pa.Mesh.bump_hex(9, 7, 5).renumbered("colour"),
        "batch": lambda: pa.Mesh.concat([pa.Mesh.bump_hex(5, 4, 3, h) for h in (0.02, 0.05)]),
    }


def run(mesh, steps, **over):
    base = dict(mach=0.5, cfl_start=2.0, cfl_end=2.0, viscous=1, reynolds=5e4, **over)
    p = pa.default_params(**base)
    s = pa.Solver(mesh, [p] * mesh.n_cases if mesh.n_cases > 1 else p)
    s.init_freestream()
    s.set_state(perturbed_state(mesh.n_total, mesh.n_cell, FREE, 5, amp=0.01))
    s.iterate(1, steps)
    return {k: s.get_field(k) for k in ("q", "res", "dq", "delta_flux")}


@pytest.mark.parametrize("name", sorted(shapes()))
def test_sweep_level_storage_equals_mesh_storage(name):
    mesh = shapes()[name]()
    a, b = run(mesh, 4, storage_order=0), run(mesh, 4, storage_order=1)
    for k in a:
        assert np.array_equal(a[k], b[k]), (name, k)
