"""The one-launch starts of a run against the state they stand for
(execution_pr.c, execution_cc.c:71-92, execution_bfs.c:70-116).

Bars: every word equal; the PageRank start is two FP64 divisions.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ONES = np.uint64(2**64 - 1)


def _words(gz, ptr, n, dtype=np.uint64):
    out = np.empty(n, dtype)
    if n:
        gz.lib.gz_copy_to_host(out.ctypes.data_as(gz.vp), gz.vp(ptr), gz.C.c_size_t(8 * n))
    return out


@pytest.mark.parametrize("relabel", [False, True])
@pytest.mark.parametrize("V", [1, 63, 64, 65, 256, 257, 4097])
def test_prepared_state(gz, device, V, relabel):
    rng = np.random.default_rng(V + 7)
    pairs = rng.integers(0, V, size=(5 * V, 2), dtype=np.uint64)
    gz.load_pairs_device(V, pairs, relabel=relabel)
    old, deg = gz.original_ids(), gz.outdegrees()
    fw = (V + 63) // 64
    G = gz.phase_graph

    for alg in ("pr", "cc", "bfs", "cc", "pr"):  # each start over another's leavings
        root = int(pairs[0, 0])
        o = gz.options(alg, root=root) if alg == "bfs" else gz.options(alg)
        gz.run(o)
        gz.lib.gz_execution_prepare(gz.C.byref(o))
        props = _words(gz, G.vertex_props, V)
        has, wants = _words(gz, G.frontier_has_info, fw), _words(gz, G.frontier_wants_info, fw)
        if alg == "pr":
            want = (1.0 / float(V)) / np.where(deg == 0, float(V), deg)  # device order
            assert np.array_equal(props.view(np.float64), want)
            assert not _words(gz, G.vertex_accumulators, V).any()
        else:
            assert not _words(gz, G.vertex_accumulators, fw).any()
        if alg == "cc":
            assert np.array_equal(props, old)
        if alg == "bfs":
            at = int(np.nonzero(old == root)[0][0])
            assert props[at] == np.uint64(2**48 - 1)
            assert np.all(np.delete(props, at) == ONES)
            bits = np.zeros(fw * 64, bool)
            bits[at] = True
            got = np.unpackbits(has.view(np.uint8), bitorder="little").astype(bool)
            assert np.array_equal(got, bits)
            free = np.unpackbits(wants.view(np.uint8), bitorder="little").astype(bool)
            assert np.array_equal(free[:V], ~bits[:V])
        else:
            assert np.all(has == ONES) and np.all(wants == ONES)
