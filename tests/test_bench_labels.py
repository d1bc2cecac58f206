"""bench.py names the kernels that took the timed steps, not those of the
profiled run beside them."""

import bench


def _path(chain, stages, launches):
    return {"chain_steps": chain, "stage_steps": stages, "chain_launches": launches, "lanes": 1}


def test_timed_steps_as_a_chain():
    timed = bench.timed_as(_path(5, 0, 20), _path(25, 0, 60))
    assert timed == {"as": "chain", "launches_per_step": 2.0}
    assert "k_chain<double" in bench.search_label(timed, "fp64", 5)
    assert "k_chain<float, 2, false, true>" in bench.search_label(timed, "mixed", 5, ensemble=True)
    kb = bench.kernel_bytes(1000, 6000, 0, 1, 500)
    e = bench.step_roofline_entry(timed, "fp64", kb, 0.5, {"force": 0.1, "search": 0.2}, {}, {}, "none.md")
    assert e["kernel"] == "k_chain<double, 2, false, false>" and e["ms"] == 0.5
    assert e["algorithmic_bytes_per_launch"] == kb["force"] + kb["walls"]


def test_timed_steps_as_stages():
    timed = bench.timed_as(_path(0, 5, 0), _path(0, 25, 0))
    assert timed == {"as": "stages", "launches_per_step": None}
    assert bench.search_label(timed, "fp64", 4) == "k_topo_half/k_topo_apply"
    kb = bench.kernel_bytes(1000, 6000, 0, 1, 500)
    e = bench.step_roofline_entry(timed, "fp64", kb, 0.5, {"force": 0.1, "search": 0.2},
                                  {"force": "k_force", "search": "k_topo_half/k_topo_apply"}, {}, "none.md")
    assert e["kernel"] == "k_topo_half/k_topo_apply" and e["ms"] == 0.2
    assert e["algorithmic_bytes_per_launch"] == kb["search"]
