"""GPU parity at the sizes where the register networks, their row classes and
the scans change path: records per vertex and VT row lengths around each
network's size and past the largest, buckets that need several placement
rounds, cell counts around a tile of the chained scan, and vertex counts
around the scan's launch forms.  Everything is integer and compared exactly
with the CPU oracle."""
import numpy as np
import pytest

from oracle import binding as O

pytestmark = pytest.mark.gpu


def fans(sizes, ring=20):
    """One centre vertex per entry of `sizes` with that many cells around it:
    (centre, a_i, a_i+1, a_i+2) along a strip of its own vertices, closed
    after `ring` of them, so degrees stay below 33 while cells per vertex
    grow.  Two fans share a vertex with their neighbours."""
    cells, n = [], 0
    for r in sizes:
        c, a0 = n, n + 1
        q = min(ring, r + 2)
        cells += [(c, a0 + i % q, a0 + (i + 1) % q, a0 + (i + 2) % q) for i in range(r)]
        n = a0 + q - 1  # the last strip vertex starts the next fan
    return np.array(cells, np.int32), n + 1


EDGES = [1, 7, 8, 9, 23, 24, 25, 31, 32, 33, 39, 40, 41, 47, 48, 49, 57, 120]


def check_vv_cp(t, cells, V, scalars, bv, route=0):
    with t.Mesh(cells, V, scalars) as m:
        m.set_config(variant=2)
        m.set_bucket(bv, 4096)
        if route:
            m.set_routing(route)
        m.vv_critpoints()
        off, vals = m.relation("VV")
        cls = m.classes()
    VV = O.vv(cells, V)
    S = VV.sorted_rows()
    assert np.array_equal(off, S.off) and np.array_equal(vals[:, 0], S.val[:, 0])
    assert np.array_equal(cls, O.critpoints(VV, np.asarray(scalars, np.float64), V))


@pytest.mark.parametrize("bv", [7, 8])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_rows_at_network_sizes(gpu, bv, dtype):
    cells, V = fans(EDGES)
    s = np.random.default_rng(5).random(V).astype(dtype)
    check_vv_cp(gpu, cells, V, s, bv)


@pytest.mark.parametrize("bv,route", [(7, 1), (7, 2), (8, 1), (8, 2)])
def test_bucket_of_several_rounds(gpu, bv, route):
    """Nearly 45 records a vertex on few neighbours: more than a bucket's slots."""
    rng = np.random.default_rng(9)
    V, T, win = 700, 7900, 12
    w0 = rng.integers(0, V - win + 1, T)
    cells = np.array([w + rng.choice(win, 4, replace=False) for w in w0], np.int32)
    check_vv_cp(gpu, cells, V, rng.random(V).astype(np.float32), bv, route)


def test_degree_around_a_mask(gpu):
    """31 to 34 neighbours: the last slot of the row and the heavy kernel."""
    cells, V = fans([29, 30, 31, 32], ring=40)
    check_vv_cp(gpu, cells, V, np.random.default_rng(2).random(V).astype(np.float32), 7)


@pytest.mark.parametrize("drop", [0, 1, 2, 255])
def test_relations_at_network_sizes(gpu, drop):
    """Every relation on fans (rows up to and past the largest network), the
    number of cells at and around multiples of a tile of 256."""
    from test_gpu_relations import check_all

    cells, V = fans(EDGES)
    rng = np.random.default_rng(drop)
    cells = np.sort(rng.permutation(V).astype(np.int32)[cells], axis=1)
    T = 512 - drop
    check_all(gpu, cells[rng.permutation(len(cells))][:T], V, expect_ft=False)


@pytest.mark.parametrize("upper", [[1, 2, 4], [13, 14, 15], [29, 30, 31], [60, 61, 62, 63], [254, 300]])
def test_edges_of_long_rows(gpu, upper):
    """Every relation on centres with that many cells, so that many + 2 upper
    neighbours; the ids of a row's edges in any order."""
    from test_gpu_relations import check_all

    cells, V = fans(upper, ring=400)
    order = np.random.default_rng(len(upper)).permutation(len(cells))
    check_all(gpu, np.ascontiguousarray(cells[order]), V, expect_ft=False)


@pytest.mark.parametrize("V", [4095, 16384, 16385, 2048 * 4096, 2048 * 4096 + 1])
def test_offsets_at_scan_forms(gpu, V):
    """A few cells spread over V vertices: the offsets come from one scan."""
    rng = np.random.default_rng(V)
    cells = np.sort(np.array([rng.choice(V, 4, replace=False) for _ in range(300)], np.int32), axis=1)
    with gpu.Mesh(cells, V) as m:
        m.build(gpu.flags("VV"))
        off, vals = m.relation("VV")
    S = O.vv(cells, V).sorted_rows()
    assert np.array_equal(off, S.off) and np.array_equal(vals[:, 0], S.val[:, 0])
