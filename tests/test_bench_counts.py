"""Query figures of the benchmark: the bytes that the statistics entry points
count are those of one lane walking alone, so they make a rate with the time of a
kernel only where its lanes walk like that (triangles), not for the point kernels,
whose lanes share their wave's subtrees."""
import bench

STATS = {"queries": 10, "node_bytes": 6400, "prims": 50}


def test_point_kernels_have_no_rate():
    c = bench.points_counts(STATS, 0.5, 20, 16, "fcp_points")
    assert c["node_bytes_per_query"] == 640 and c["prims_per_query"] == 5 and c["avg_launch_ms"] == 0.5
    assert not {"achieved", "frac", "peak", "bound"} & set(c)


def test_triangle_kernel_has_one():
    c = bench.query_roofline(STATS, 0.5, 20, 52, "fcp_triangles")
    assert c["bytes_per_query"] == 20 + 640 + 5 * 52
    assert abs(c["achieved"] - c["bytes_per_launch"] / 0.5e-3 / 1e9) < 1e-9 * c["achieved"]
