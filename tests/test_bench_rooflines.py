"""The per-kernel rooflines that bench.py reports: cells, time and measured traffic of a class
belong to the launches of that class."""
import bench


def test_elastic_classes_of_both_step_forms():
    names = [n for _, n in bench.KERNEL_CLASSES[True]]
    assert [k for k, _ in bench.KERNEL_CLASSES[True]] == [0, 5, 1, 3]
    out = bench.kernel_rooflines(True, 200, 200, 200, {n: 100.0 for n in names}, 200)
    assert list(out) == names
    assert [out[n]["cells"] for n in names] == [200 * 200 * k for k in (200, 188, 16, 12)]
    assert [out[n]["traffic_bytes"] for n in names] == [859156480, 411527783 + 324555981, 38142056, 202203417]
    # a forward step of the several-launch form and an adjoint step of one launch
    assert 2 * bench.measured_traffic(200) == sum(out[n]["traffic_bytes"] for n in names) // 2 * 2
