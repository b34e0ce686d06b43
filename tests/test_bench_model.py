"""The byte models of bench.py (no GPU): the build roofline is a rate of one
build, and the query bytes are ones that the query reads."""
import numpy as np

import bench

ST = {"actives": 10, "edges": 1000, "tails": 100, "dq_labels": 5000, "labels_appended": 400,
      "ms_push": 2.0, "n_push": 4, "ms_add": 1.0, "n_add": 3}


def test_build_roofline_is_of_one_build():
    r = bench.build_roofline(ST, "events", None, "rmat20_ef16")
    own = 8 * 10 + 4 * 1000 + bench.BP_RECORD_BYTES * 100
    assert r["kernel"] == "k_push" and r["launches"] == 4 and r["traffic"] is None
    assert r["alg_bytes_per_launch"] == round(own / 4, 1)
    assert r["achieved"] == round(own / 2e-3 / 1e9, 2)
    # every count of the same build, in whichever kernel dominates
    a = bench.build_roofline(dict(ST, ms_add=8.0), "events", None, "rmat20_ef16")
    assert a["kernel"] == "k_add" and a["achieved"] == round(5 * 5400 / 8e-3 / 1e9, 2)
    assert ST["ms_push"] == 2.0 and set(ST) == {"actives", "edges", "tails", "dq_labels", "labels_appended",
                                                "ms_push", "n_push", "ms_add", "n_add"}


def test_traffic_belongs_to_the_workload():
    tr = {"workload": "rmat20_ef16", "source": "x", "kernels": {"k_push": {"bytes_per_launch": 7}}}
    assert bench.build_roofline(ST, "events", tr, "rmat20_ef16")["traffic"] == 7
    assert bench.build_roofline(ST, "events", tr, "rmat18_ef16")["traffic"] is None


def test_query_bytes():
    # (ids and answer of 3 pairs; two connected ones with 5 + 7 and 0 + 1 labels)
    got = bench.query_bytes(np.array([True, False, True]), [5, 9, 0], [7, 9, 1])
    assert got == 3 * 9 + 2 * 16 + (256 + 4 * 12) + (256 + 4 * 1)
