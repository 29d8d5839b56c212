"""Meshes with long rows on the CPU kernel emulator (AddressSanitizer, exact
allocations), against the oracle: the parts of the relation builds that only
vertices with many cells or neighbours reach.  No GPU is needed.
"""
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

import pytest

from test_emu_kernels import EMU, emu_env  # noqa: F401  (fixture)

CASES = [
    # more neighbours than a kernel holds, the hub with the highest or the
    # lowest id, in the bucketed and the vertex-lane form
    ("capacity", 0, 2), ("capacity", 1, 2), ("capacity", 0, 1), ("capacity", 1, 1),
    # rows beyond the join networks, alone in a wave and beside short ones
    ("hub_rows", 50, 0, 0, 0), ("hub_rows", 20, 33, 10, 1), ("hub_rows", 30, 20, 0, 1, 1),
    # a vertex's faces by the wave, an edge's by the wave and by the block
    ("hub_rows", 1, 100, 0, 1), ("hub_rows", 70, 1, 0, 1),
    # VV and classes of vertices with many cells
    ("heavy", 0), ("heavy", 1), ("heavy", 2),
    # a vertex's edges ordered by the whole block
    ("vertex_rows", 127, 1), ("vertex_rows", 140, 0),
]


@pytest.fixture(scope="module")
def results(emu_env):  # noqa: F811
    def run(case):
        return subprocess.run([sys.executable, str(EMU / "run_case.py"), *map(str, case)],
                              env=emu_env, capture_output=True, text=True, timeout=600)

    with ThreadPoolExecutor(6) as ex:
        return dict(zip(CASES, ex.map(run, CASES)))


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_long_rows(results, case):
    r = results[case]
    assert r.returncode == 0 and "ok " in r.stdout, (r.stdout + r.stderr)[-4000:]
