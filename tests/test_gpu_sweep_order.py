"""Storage in sweep-level order and the dataflow sweeps over it, at the shapes
where an order or a chunk can go wrong: one cell, levels of exactly 64 and of
65 cells, one-cell levels, a random numbering (many short levels), a colour
numbering (two levels of half the mesh, six lower neighbours), wide ones past
the quad form's limit of cells per level, a batch.  Every comparison is bitwise:
the order only moves where a cell's data live."""
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
        "two_wide_levels": lambda: pa.Mesh.bump_hex(101, 60, 7).renumbered("colour"),
        "batch": lambda: pa.Mesh.concat([pa.Mesh.bump_hex(5, 4, 3, h) for h in (0.02, 0.05)]),
    }


def run(mesh, steps, **over):
    base = dict(dict(mach=0.5, cfl_start=2.0, cfl_end=2.0, viscous=1, reynolds=5e4), **over)
    p = pa.default_params(**base)
    s = pa.Solver(mesh, [p] * mesh.n_cases if mesh.n_cases > 1 else p)
    s.init_freestream()
    s.set_state(perturbed_state(mesh.n_total, mesh.n_cell, FREE, 5, amp=0.01))
    s.iterate(1, steps)
    return {k: s.get_field(k) for k in ("q", "res", "dq", "delta_flux") + (("nut", "dq_t") if over.get("viscous") == 3 else ())}


@pytest.mark.parametrize("name", sorted(shapes()))
def test_sweep_level_storage_equals_mesh_storage(name):
    mesh = shapes()[name]()
    a, b = run(mesh, 4, storage_order=0), run(mesh, 4, storage_order=1)
    for k in a:
        assert np.array_equal(a[k], b[k]), (name, k)


@pytest.mark.parametrize("form", [0, 2, 3])
@pytest.mark.parametrize("name", sorted(shapes()))
def test_dataflow_sweep_at_chunk_edges_equals_level_form(name, form):
    mesh = shapes()[name]()
    a, b = run(mesh, 4, sweep_form=form), run(mesh, 4, sweep_form=1)
    for k in a:
        assert np.array_equal(a[k], b[k]), (name, k)


@pytest.mark.parametrize("name,over", [(n, o) for n in sorted(shapes()) for o in (
    {}, dict(viscous=3, cfl_start=0.5, cfl_end=0.5), dict(n_lusgs_sweeps=3)) if n != "batch" or not o])
def test_level_form_in_mesh_order(name, over):
    """Increments as rows of one line each instead of planes (a batch is laminar,
    with one sweep pair)."""
    mesh = shapes()[name]()
    a, b = run(mesh, 4, sweep_form=1, storage_order=1, **over), run(mesh, 4, **over)
    for k in a:
        assert np.array_equal(a[k], b[k]), (name, k)


@pytest.mark.parametrize("form", [0, 2])
@pytest.mark.parametrize("name", ["levels_of_65", "hex_coloured", "two_wide_levels"])
def test_carried_turbulence_sweep_at_chunk_edges(name, form):
    mesh = shapes()[name]()
    a, b = (run(mesh, 4, sweep_form=f, viscous=3, cfl_start=0.5, cfl_end=0.5) for f in (form, 1))
    for k in a:
        assert np.array_equal(a[k], b[k]), (name, k)


@pytest.mark.parametrize("name", ["hex_coloured", "two_wide_levels"])
def test_mixed_form_at_chunk_edges(name):
    mesh = shapes()[name]()
    a, b = run(mesh, 4, sweep_form=0, precision=1), run(mesh, 4, sweep_form=1, precision=1)
    for k in a:
        assert np.array_equal(a[k], b[k]), (name, k)


def wide_cell_mesh(wide_first):
    """Two columns of 3x3 unit cells' worth of space: one 1x3x3 polyhedron
    whose inner side is nine faces, and nine unit hexahedra.  Numbered first, the polyhedron
    has nine higher neighbours (a backward sweep too wide for the dataflow
    form, a forward one that is not); numbered last, nine lower ones."""
    xs = [(i, j, k) for i in range(3) for j in range(4) for k in range(4)]
    node = {p: n for n, p in enumerate(xs)}
    quad = lambda pts: [node[p] for p in pts]
    big, small = (0, 1) if wide_first else (9, 0)
    cell = lambda j, k: small + 3 * k + j
    bnd, inner = [], []
    ring = [(0, j, 0) for j in range(4)] + [(0, 3, k) for k in range(1, 4)] + [(0, j, 3) for j in (2, 1, 0)] + \
           [(0, 0, k) for k in (2, 1)]
    bnd.append((quad(ring)[::-1], big))
    for j in range(3):  # the polyhedron's own y and z sides
        bnd.append((quad([(0, j, 0), (1, j, 0), (1, j + 1, 0), (0, j + 1, 0)])[::-1], big))
        bnd.append((quad([(0, j, 3), (1, j, 3), (1, j + 1, 3), (0, j + 1, 3)]), big))
        bnd.append((quad([(0, 0, j), (0, 0, j + 1), (1, 0, j + 1), (1, 0, j)])[::-1], big))
        bnd.append((quad([(0, 3, j), (0, 3, j + 1), (1, 3, j + 1), (1, 3, j)]), big))
    for k in range(3):
        for j in range(3):
            x = lambda i: quad([(i, j, k), (i, j + 1, k), (i, j + 1, k + 1), (i, j, k + 1)])
            a, b = (big, cell(j, k)) if wide_first else (cell(j, k), big)
            inner.append((x(1) if wide_first else x(1)[::-1], a, b))
            bnd.append((x(2), cell(j, k)))
            y = lambda jj: quad([(1, jj, k), (1, jj, k + 1), (2, jj, k + 1), (2, jj, k)])
            z = lambda kk: quad([(1, j, kk), (2, j, kk), (2, j + 1, kk), (1, j + 1, kk)])
            if j == 0: bnd.append((y(0)[::-1], cell(j, k)))
            if j == 2: bnd.append((y(3), cell(j, k)))
            else: inner.append((y(j + 1), cell(j, k), cell(j + 1, k)))
            if k == 0: bnd.append((z(0)[::-1], cell(j, k)))
            if k == 2: bnd.append((z(3), cell(j, k)))
            else: inner.append((z(k + 1), cell(j, k), cell(j, k + 1)))
    nodes = {big: sorted({n for f, *cs in bnd + inner if big in cs for n in f})}
    for j in range(3):
        for k in range(3):
            nodes[cell(j, k)] = [node[(i, j + a, k + b)] for i in (1, 2) for a in (0, 1) for b in (0, 1)]
    faces = [f for f, *_ in bnd + inner]
    return pa.Mesh.from_arrays(
        *np.array(xs, float).T, np.cumsum([0] + [len(f) for f in faces]), np.concatenate(faces),
        [c for _, c in bnd] + [a for _, a, _ in inner], [10 + n for n in range(len(bnd))] + [b for *_, b in inner],
        len(bnd), [pa.BC["farfield"]] * len(bnd), np.cumsum([0] + [len(nodes[c]) for c in range(10)]),
        np.concatenate([nodes[c] for c in range(10)]))


@pytest.mark.parametrize("wide_first", [True, False])
def test_one_direction_in_dataflow_form_the_other_by_level(wide_first):
    mesh = wide_cell_mesh(wide_first)
    met = mesh.metrics()
    assert met["vol"][:10].min() > 0 and abs(met["vol"][:10].sum() - 18.0) < 1e-12
    a, b = run(mesh, 5, sweep_form=0), run(mesh, 5, sweep_form=1)
    for k in a:
        assert np.array_equal(a[k], b[k]), k


@pytest.mark.parametrize("wide_first", [True, False])
def test_level_form_of_wide_cells_in_mesh_order(wide_first):
    mesh = wide_cell_mesh(wide_first)
    a, b = run(mesh, 5, sweep_form=1, storage_order=1), run(mesh, 5, sweep_form=1)
    for k in a:
        assert np.array_equal(a[k], b[k]), k


@pytest.mark.parametrize("wide_first", [True, False])
def test_graphs_with_one_direction_in_dataflow_form(wide_first):
    """A step then swaps the two increment buffers once, so that eight-step
    graphs start from either assignment: replays after odd numbers of steps
    and after a hook's sweep equal eager launches of the level form."""
    mesh = wide_cell_mesh(wide_first)
    p = [pa.default_params(mach=0.5, cfl_start=2.0, cfl_end=2.0, viscous=1, reynolds=5e4, sweep_form=f) for f in (0, 1)]
    a, b = (pa.Solver(mesh, q) for q in p)
    b.set_launch_mode("eager")
    step = 1
    for s in (a, b):
        s.init_freestream()
        s.set_state(perturbed_state(mesh.n_total, mesh.n_cell, FREE, 5, amp=0.01))
    for n in (8, 3, 17, 1, 24):
        assert np.array_equal(a.iterate(step, n), b.iterate(step, n)), n
        step += n
        for s in (a, b):
            s.residual()
            s.spectrum_radius()
            s.time_step(step)
            s.lusgs()
        step += 1
        for k in ("q", "res", "dq", "delta_flux"):
            assert np.array_equal(a.get_field(k), b.get_field(k)), (n, k)
    assert a.launch_counts()[0] >= 6


def wide_levels(slots, count):
    """One mesh of `count` disconnected blocks, so that a level holds a level of
    every block: 27 cells in 7 levels with at most three swept neighbours, or 36
    cells in 6 levels with four (two i-planes exchanged, so that one has both
    its i-neighbours before it and the other both after it)."""
    if slots == 3:
        part = pa.Mesh.bump_hex(3, 3, 3)
    else:
        i, jk = np.arange(36) % 4, np.arange(36) // 4
        part = pa.Mesh.bump_hex(4, 3, 3).renumbered("perm", 4 * jk + np.array([0, 2, 1, 3])[i])
    c = pa.Mesh.concat([part] * count).connectivity()
    return pa.Mesh.from_arrays(c["x"], c["y"], c["z"], c["face_node_ptr"], c["face_nodes"], c["left"], c["right"],
                               c["n_bface"], c["bc_type"], c["cell_node_ptr"], c["cell_nodes"])


WIDE = {3: 4667, 4: 3001}  # blocks: just past 18,000 cells per level
INVISCID, TURBULENT = dict(viscous=0, reynolds=0.0), dict(viscous=3, cfl_start=0.5, cfl_end=0.5)


@pytest.mark.parametrize("slots,count,form,over", [
    (3, WIDE[3], 0, INVISCID), (3, WIDE[3], 0, dict(precision=1)), (3, WIDE[3], 0, TURBULENT), (3, WIDE[3], 2, {}),
    (3, WIDE[3], 3, TURBULENT), (4, WIDE[4], 0, INVISCID), (4, WIDE[4], 0, dict(precision=1)),
    (4, WIDE[4], 0, TURBULENT), (4, WIDE[4], 2, TURBULENT), (4, WIDE[4], 3, {}),
    (4, 3000, 0, TURBULENT),  # at the limit: four lanes per cell
])
def test_wide_levels_with_64_cells_per_wavefront(slots, count, form, over):
    mesh = wide_levels(slots, count)
    fwd, bwd = pa.Solver(mesh, pa.default_params()).sweep_levels()
    assert fwd == bwd == {3: 7, 4: 6}[slots]
    assert (mesh.n_cell > 18000 * fwd) == (count != 3000)
    a, b = run(mesh, 4, sweep_form=form, **over), run(mesh, 4, sweep_form=1, **over)
    for k in a:
        assert np.array_equal(a[k], b[k]), k


def test_wide_levels_of_a_batch():
    """The same blocks as cases with their own Mach numbers."""
    mesh = pa.Mesh.concat([pa.Mesh.bump_hex(3, 3, 3)] * WIDE[3])
    out = []
    for form in (0, 1):
        s = pa.Solver(mesh, [pa.default_params(mach=0.3 + 0.0001 * k, cfl_start=5.0, cfl_end=5.0, precision=1,
                                               sweep_form=form) for k in range(WIDE[3])])
        s.init_freestream()
        out.append((s.iterate(1, 10), s.get_state(), s.get_field("dq")))
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("bits", [0xFFFFFFFFFFFFFFFF, 0x7FF8000000000000])
@pytest.mark.parametrize("name", ["levels_of_65", "two_wide_levels"])  # 16 and 64 cells per wavefront
def test_not_a_number_in_the_state_is_no_mark(name, bits):
    """A NaN of the caller's whose bits are those of the mark of an increment that
    is not there yet: sweeps must not wait for it (the wait bound would be
    reported), and spread it as the level form does."""
    mesh = shapes()[name]()
    q = perturbed_state(mesh.n_total, mesh.n_cell, FREE, 5, amp=0.01)
    q[:, mesh.n_cell // 3] = np.array([bits], np.uint64).view(np.float64)[0]
    out = []
    for form in (0, 1):
        s = pa.Solver(mesh, pa.default_params(mach=0.5, cfl_start=2.0, cfl_end=2.0, viscous=1, reynolds=5e4,
                                              sweep_form=form))
        s.init_freestream()
        s.set_state(q)
        s.residual()
        s.spectrum_radius()
        s.time_step(1)
        s.lusgs()
        out.append([s.get_field(k) for k in ("dq", "delta_flux", "q")])
    assert np.isnan(out[0][0]).any()
    for a, b in zip(*out):
        assert np.array_equal(a, b, equal_nan=True)
