"""GPU parity where vertices have many cells and neighbours: rows that the
joins' networks do not take and that a whole wave orders or merges.  Everything
is integer and compared exactly with the CPU oracle."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def hub_mesh(n, apart, between):
    """`n` cells (a, b, s_i, s_i+1) around the edge of two hubs, `apart` cells
    around each hub alone, and `between` cells of a strip that touches
    neither; the hubs' shared cells come among the others at regular places."""
    cells = [(0, 1, 2 + i, 3 + i) for i in range(n)]
    v = n + 3
    for hub in (0, 1):
        cells += [(hub, v + i, v + i + 1, v + i + 2) for i in range(apart)]
        v += apart + 2 if apart else 0
    strip = [(v + i, v + i + 1, v + i + 2, v + i + 3) for i in range(between)]
    v += between + 3 if between else 0
    cells = cells + strip
    order = np.argsort(np.arange(len(cells)) * 7 % max(len(cells), 1), kind="stable")
    return np.array(cells, np.int32)[order], v


def check_hubs(t, shared, apart, between, order, variant=0):
    """order 0: as hub_mesh gives it; else random cells and ids by that seed."""
    from test_gpu_relations import check_all

    cells, V = hub_mesh(shared, apart, between)
    if order:
        rng = np.random.default_rng(order)
        ids = rng.permutation(V).astype(np.int32)
        cells = np.ascontiguousarray(np.sort(ids[cells], axis=1)[rng.permutation(len(cells))])
    check_all(t, cells, V, variant, expect_ft=False)


def test_hub_rows_vertex_lane(gpu):
    """VV from the form that does not count the vertices of many cells."""
    check_hubs(gpu, 46, 30, 200, 1, variant=1)
    check_hubs(gpu, 5, 20, 200, 1, variant=1)


@pytest.mark.parametrize("order", [0, 1])
@pytest.mark.parametrize("shared,apart,between", [
    (50, 0, 0), (1000, 0, 0),            # the same long row twice
    (300, 900, 700), (1, 65, 0),         # stretches of one hub alone
    (49, 0, 64), (46, 3, 200),           # a few long rows in a wave of short ones
    (1, 4000, 0),                        # near the most neighbours a kernel holds
])
def test_hub_rows(gpu, shared, apart, between, order):
    check_hubs(gpu, shared, apart, between, order)


def seconds(t, cells, V, first, then):
    """The shortest of five builds of `then` on meshes that hold `first`."""
    best = float("inf")
    for _ in range(5):
        with t.Mesh(cells, V) as m:
            m.build(t.flags(*first.split(",")))
            m.shape(first.split(",")[0])
            t0 = time.perf_counter()
            m.build(t.flags(then))
            m.shape(then)
            best = min(best, time.perf_counter() - t0)
    return best


@pytest.mark.parametrize("first,then,n", [("VT", "TT", 34), ("TE", "EE", 44), ("VV,VT", "TE", 44)])
def test_long_rows_cost_their_entries(gpu, first, then, n):
    """4000 cells around one vertex in random order give about as many entries as
    a grid of n^3 cubes and take no more than 20 times as long (both take 0.1 to
    0.2 ms; a row's merge that starts anew for every window of a wave's output
    takes hundreds of times as long, one lane's sort by insertion thousands).  The
    fan's TE is small, 0.5 ms; one lane that searches the vertex's row for each
    of its cells takes 16."""
    i = np.random.default_rng(4).permutation(4000).astype(np.int32)
    fan = np.ascontiguousarray(np.stack([i, i + 1, i + 2, np.full(4000, 4002, np.int32)], 1))
    m = gpu.kuhn(n, seed=1)
    long = seconds(gpu, fan, 4003, first, then)
    short = seconds(gpu, m.cells, m.n_points, first, then)
    print(f"{then}: long rows {1e6 * long:.0f} us, short rows {1e6 * short:.0f} us", flush=True)
    assert long < 20 * short


HEAVY = [([46, 47, 48, 49, 50, 59, 60, 61], 20),   # cells around the row kernel's limit
         ([29, 30, 31, 48, 61, 62, 63, 64], 80),   # 31 to 33 and 63 to 66 neighbours
         ([126, 127, 128, 129, 130, 300], 30)]     # records that one wave takes, and more


def check_heavy(t, sizes, ring, dtype, seed=3):
    from test_gpu_networks import check_vv_cp, fans

    cells, V = fans(sizes, ring)
    rng = np.random.default_rng(seed)
    check_vv_cp(t, cells, V, rng.random(V).astype(dtype), 7)
    check_vv_cp(t, cells, V, rng.integers(0, 3, V).astype(dtype), 8)  # ties


@pytest.mark.parametrize("sizes,ring", HEAVY)
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_vertices_of_many_cells(gpu, sizes, ring, dtype):
    """VV and classes of the vertices that the row kernel leaves to the heavy one."""
    check_heavy(gpu, sizes, ring, dtype)


def test_many_vertices_of_many_cells_cost(gpu):
    """With every second cell of a grid split, a tenth of the vertices have 49 to
    60 cells and 27 to 32 neighbours: 2.5 times the cells, 3.6 times the time
    (41 times with a workgroup for each of them)."""
    def run(m):
        with gpu.Mesh(m.cells, m.n_points, m.scalars) as d:
            best = float("inf")
            for _ in range(6):
                t0 = time.perf_counter()
                d.vv_critpoints()
                d.shape("VV")
                best = min(best, time.perf_counter() - t0)
        return best

    plain, split = run(gpu.kuhn(48, seed=3)), run(gpu.kuhn(48, seed=3, split_fraction=0.5))
    print(f"split {1e6 * split:.0f} us, plain {1e6 * plain:.0f} us", flush=True)
    assert split < 10 * plain
