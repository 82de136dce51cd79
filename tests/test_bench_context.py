"""The reference's published A100 latencies that bench.py prints beside its own
reference-shape figures must equal the reference's result files:
results/FINAL_flexattention.csv (the S = 2048 benchmark, extra_bench.py:83-157)
and results/FINAL_seqsweep.csv (the sequence sweep, extra_bench.py:166-201),
where a sweep row counts only if its status is "generalises".  Skipped where the
reference tree is absent (it never travels to the GPU box)."""
import csv
import importlib.util
import shutil
import subprocess
from pathlib import Path

import pytest

from chia_proj_amd.workloads import REFERENCE_SWEEP_S, reference_suite

REPO = Path(__file__).resolve().parent.parent
RESULTS = Path("/root/reference/results")


def _bench():
    spec = importlib.util.spec_from_file_location("bench_under_test", REPO / "bench.py")
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def _rows(name):
    path = RESULTS / name
    if not path.is_file():
        pytest.skip(f"{path} not present")
    with open(path, newline="") as fh:
        return list(csv.DictReader(fh))


def _num(x):
    return float(x) if x not in ("", None) else None


def test_flexattention_table_matches_reference_file():
    bench = _bench()
    rows = {r["op"]: r for r in _rows("FINAL_flexattention.csv")}
    assert set(bench.A100_PUBLISHED_US) == set(rows) == {c.op for c in reference_suite()}
    for op, (gs, flex) in bench.A100_PUBLISHED_US.items():
        assert gs == _num(rows[op]["graphsynth_us"]), op
        assert flex == _num(rows[op]["flex_us"]), op


def test_seqsweep_table_matches_reference_file():
    bench = _bench()
    rows = _rows("FINAL_seqsweep.csv")
    assert {int(r["S"]) for r in rows} == set(REFERENCE_SWEEP_S)
    assert set(bench.A100_SEQSWEEP_US) == {c.op for c in reference_suite()}
    for r in rows:
        want = _num(r["graphsynth_us"]) if r["status"] == "generalises" else None
        assert bench.A100_SEQSWEEP_US[r["op"]][int(r["S"])] == want, (r["op"], r["S"], r["status"])


def test_reference_suites_keep_the_reference_shape():
    for S in REFERENCE_SWEEP_S:
        cases = reference_suite(S)
        assert [c.op for c in cases] == [c.op for c in reference_suite()]
        assert all((c.B, c.H, c.S, c.D) == (2, 32, S, 128) and c.params == {} for c in cases)
    assert reference_suite()[0].seed == 20262048  # the benchmark's draw is unchanged


@pytest.mark.skipif(shutil.which("nm") is None, reason="nm not available")
def test_kernel_names_are_the_librarys():
    """The instantiation names that bench.py looks recorded HBM traffic up by are kernels of the
    built library, as rocprofv3 prints them, and profiles/traffic.json records those names."""
    from chia_proj_amd import _lib
    from chia_proj_amd.workloads import headline_suite, north_star_suite

    if not Path(_lib.LIB_PATH).exists():
        pytest.skip("the library is not built")
    out = subprocess.run(["nm", "-C", str(_lib.LIB_PATH)], capture_output=True, text=True, check=True).stdout
    names = {line.split(" ", 2)[2] for line in out.splitlines() if "chia::attn_fwd" in line}
    bench = _bench()
    for suite, cases in (("headline", headline_suite()), ("northstar", north_star_suite())):
        for c in cases:
            params = dict(c.params, temperature=[1.0] * c.H) if c.temperature else c.params
            name = bench.kernel_name(c.op, c.B, c.H, c.S, c.D, params)
            assert name in names, (c.name, name)
            assert bench.load_traffic(suite, c.op, name), (c.name, name)
