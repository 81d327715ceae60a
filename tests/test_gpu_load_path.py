"""Loads and read-backs: copies through the staging chunks, the endpoint check
on the uploaded pairs, and buffers handed out again after a release.

Bars: bytes equal; the same message and exit status for a bad endpoint.
"""
import pathlib
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CHUNK = 2 << 20  # a staging chunk; copies of two chunks and more are staged


@pytest.mark.parametrize("size", [8, 2 * CHUNK - 1, 2 * CHUNK, 2 * CHUNK + 1, 3 * CHUNK, 5 * CHUNK + 4093])
def test_copies_at_chunk_edges(gz, device, size):
    src = np.random.default_rng(size).integers(0, 256, size=size + 1, dtype=np.uint8)[1:]  # odd address
    dst = np.zeros(size + 9, np.uint8)
    gz.lib.gz_device_malloc.restype = gz.vp
    d = gz.vp(gz.lib.gz_device_malloc(gz.C.c_size_t(size)))
    try:
        gz.lib.gz_copy_to_device(d, src.ctypes.data_as(gz.vp), gz.C.c_size_t(size))
        gz.lib.gz_copy_to_host(dst[1:].ctypes.data_as(gz.vp), d, gz.C.c_size_t(size))
    finally:
        gz.lib.gz_device_free(d)
    assert np.array_equal(dst[1 : size + 1], src)
    assert dst[0] == 0 and not dst[size + 1 :].any()


def test_graphs_of_other_sizes_share_buffers(gz, device):
    # blocks of a released graph serve the next one, also a smaller one
    def answers(V, seed):
        pairs = np.random.default_rng(seed).integers(0, V, size=(6 * V, 2), dtype=np.uint64)
        gz.load_pairs_device(V, pairs, relabel=True)
        gz.run(gz.options("cc"))
        labels = gz.cc_labels().copy()
        gz.run(gz.options("pr", iterations=4))
        return labels, gz.pr_ranks().copy()

    sizes = [(30011, 1), (29000, 2), (517, 3), (70001, 4), (30011, 1)]
    first = {}
    for V, seed in sizes + sizes:
        got = answers(V, seed)
        want = first.setdefault((V, seed), got)
        assert np.array_equal(got[0], want[0])
        assert np.allclose(got[1], want[1], rtol=1e-12, atol=0)
    

@pytest.mark.parametrize("at", [0, 1, 2 * 999 + 1])
def test_bad_endpoint_ends_the_process(gz, device, at):
    # the bad endpoint with the smallest index is the one named
    code = f"""
import sys
sys.path.insert(0, {str(pathlib.Path(gz.__file__).parent)!r})
import numpy as np, grazelle as gz
pairs = np.arange(2000, dtype=np.uint64).reshape(-1, 2) % np.uint64(77)
words = pairs.reshape(-1)
words[{at}] = 77
words[{at} + 1 :: 5] = 999
gz.load_pairs_device(77, pairs)
print("loaded")
"""
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert r.returncode == 65
    assert "edge endpoint 77 is not below V = 77" in r.stderr
    assert "loaded" not in r.stdout


def _in_a_process(gz, body):
    """Runs body in a process of its own, after a load of R-MAT s23 whose
    temporaries (two arrays of 2^27 words and more) leave the pool idle blocks;
    free() is the device's free memory."""
    code = f"""
import sys, torch
sys.path.insert(0, {str(pathlib.Path(gz.__file__).parent)!r})
import grazelle as gz
gz.init()
free = lambda: torch.cuda.mem_get_info()[0]
gz.load_rmat_device(10, 16 << 10, 1)
before = free()
gz.load_rmat_device(23, 16 << 23, 1)
{body}
print("done")
"""
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "done" in r.stdout, r.stderr


def test_allocation_takes_back_idle_blocks(gz, device):
    # a request beyond what is free, by less than the idle blocks hold
    _in_a_process(gz, """
gz.lib.gz_device_malloc.restype, gz.lib.gz_device_malloc.argtypes = gz.vp, [gz.C.c_size_t]
gz.lib.gz_device_free.argtypes = [gz.vp]
gz.lib.gz_device_free(gz.lib.gz_device_malloc(free() + (512 << 20)))
""")


def test_release_gives_idle_blocks_back(gz, device):
    # what stays is the scratch of the larger graph (by its 2^23 vertices)
    _in_a_process(gz, """
gz.release()
assert before - free() < 512 << 20, (before, free())
""")


def test_mirrors_asked_for_by_several_threads(gz, device):
    # the first requests for the out-degrees and the id map come at once
    import threading

    n, V = 8, 1 << 20
    for seed in range(4):
        gz.load_rmat_device(20, 4 << 20, seed, relabel=True)
        go, got = threading.Barrier(n), [None] * n
        last = gz.original_ids()[-64:]

        def ask(i):
            go.wait()
            ids = [gz.lib.gz_graph_device_vertex(int(v)) for v in last] if i % 2 else None
            p = gz.lib.gz_graph_outdegrees_host()
            got[i] = (gz.C.addressof(p.contents), ids,
                      np.ctypeslib.as_array(p, shape=(V,)).sum())

        threads = [threading.Thread(target=ask, args=(i,)) for i in range(n)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert len({g[0] for g in got}) == 1
        assert all(g[2] == gz.num_edges() for g in got)
        assert all(g[1] in (None, list(range(V - 64, V))) for g in got)


def test_small_loads_after_a_large_one_reuse_their_blocks(gz, device):
    # the blocks of a graph that fills the pool make room for smaller loads':
    # the third of them makes no device allocation and no free
    gz.lib.gz_pool_device_calls.restype = gz.C.c_uint64
    gz.load_rmat_device(24, 16 << 24, 1)
    calls = []
    for seed in range(4):
        gz.load_rmat_device(20, 16 << 20, 1, relabel=True)
        gz.run(gz.options("pr", iterations=2))
        gz.pr_ranks()
        calls.append(gz.lib.gz_pool_device_calls())
    assert calls[2] == calls[1] and calls[3] == calls[2], calls
    gz.release()
    assert gz.lib.gz_pool_device_calls() > calls[-1]
