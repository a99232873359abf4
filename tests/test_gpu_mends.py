"""Calls whose buffers, counters or routes an earlier call of the same forest left behind."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PUTS = {"2phase": "puts_2phase_with_valuehp", "latching": "puts_latching_with_valuehp_v2"}


def _put(t, b, mode="2phase"):
    targets, n = getattr(t, PUTS[mode])(b)
    t.hash_onepass_v2(targets, n)
    return t.get_root_hash()


def _random_batch(workloads, rng, n):
    flat, lens = workloads.random_values(rng, n, 1, 60)
    return workloads.batch_from_fixed(workloads.unique_random_keys(rng, n, 32), flat, lens)


@pytest.mark.parametrize("between", ["gets", "insert", "latching", "values", "export"])
def test_graph_is_captured_again_after_a_buffer_moved(gmpt, workloads, oracle, between):
    # a capture holds the addresses of the workspaces and pools: a larger call
    # between two rebuilds replaces some of them
    rng = np.random.default_rng(len(between))
    small, large = _random_batch(workloads, rng, 2000), _random_batch(workloads, rng, 150_000)
    want = oracle.root_of(small)
    db = gmpt.DeviceBatch(small, adopt_values=True)
    t = gmpt.MPT(device=0)
    assert t.rebuild_graph(db) is False
    assert t.rebuild_graph(db) is True and t.get_root_hash() == want
    if between == "gets":
        assert (t.gets_parallel(large)[1] == t.gets_parallel(large.subset([0]))[1][0]).all()
    elif between == "values":
        assert t.get_values(large.subset(range(60_000)))[:3] == t.get_values(large.subset(range(3)))
    elif between == "export":
        assert len(t.flush_dirty_nodes(large)) > 0
    else:
        _put(t, large, "latching" if between == "latching" else "2phase")
    # (an export of few nodes has workspaces of its own)
    assert t.rebuild_graph(db) is (between == "export") and t.get_root_hash() == want
    for _ in range(2):
        assert t.rebuild_graph(db) is True and t.get_root_hash() == want
    got, sizes = t.gets_parallel(small)
    assert (sizes == np.diff(small.values_indexs.reshape(-1, 2), axis=1).ravel() + 1).all()
    t.close()
    db.free()
