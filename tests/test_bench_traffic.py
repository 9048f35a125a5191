"""bench.py divides counted HBM bytes only by the time of the bins that they
were counted with."""

import bench


def test_c4_traffic_needs_the_counted_bins():
    (bins, p, th), counted = next(iter(bench.TRAFFIC_BYTES_C4.items()))
    info = {"bin_size": bins + (1,), "max_points": p, "threads": th}
    got = bench.c4_traffic(info, 1e9, 1.0, 2.0)
    assert got["c4_traffic_over_algorithmic"]["spread"] == round(counted["spread"] / 1e9, 2)
    assert got["c4_hbm_GBps_measured_traffic"] == {"interp": round(counted["interp"] / 1e6, 1),
                                                   "spread": round(counted["spread"] / 2e6, 1)}
    for other in ({"bin_size": (32, 32, 1)}, {"max_points": p // 4}, {"threads": 128}):
        got = bench.c4_traffic(dict(info, **other), 1e9, 1.0, 2.0)
        assert got["c4_traffic_over_algorithmic"] is None and got["c4_hbm_GBps_measured_traffic"] is None
