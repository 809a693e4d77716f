"""bench.py's HBM bytes per step from a profiler's counter files: the two sweeps
of a step may be launches of one kernel or of two."""
import pytest

import bench


def write(path, rows):
    path.mkdir()
    lines = ["Kernel_Name,Counter_Name,Counter_Value"]
    lines += [f'"void phl::{k}(phl::DevMesh, int)",FETCH_SIZE,{v}' for k, v in rows]
    (path / "pass_counter_collection.csv").write_text("\n".join(lines))
    return bench._counter_means(str(path))


@pytest.mark.parametrize("names", [("k_sweep_flow<1, true>", "k_sweep_flow<1, true>"),
                                   ("k_sweep_flow<3, false>", "k_sweep_flow<6, false>")])
def test_sweep_traffic_is_of_both_directions(tmp_path, names):
    n = bench.TRAFFIC_STEPS
    means = write(tmp_path / "p", [(names[0], 100.0)] * n + [(names[1], 300.0)] * n + [("k_face_flux<double>", 7.0)] * n)
    kernels = {k: {c: v} for (k, c), (v, _) in means.items()}
    tr = dict(kernels=kernels, per_step={k: m / n for (k, _), (_, m) in means.items()})
    assert bench.step_traffic(tr, ("k_sweep_flow",)) == 400.0
    assert bench.step_traffic(tr, ("k_face_flux",)) == 7.0
    assert bench.step_traffic(tr, ("k_other",)) is None
