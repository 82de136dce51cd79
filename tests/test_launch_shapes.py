"""CPU checks of what chia_attn_fwd and chia_attn_bwd launch (tests/cpp/launch_shapes.cpp: the
C ABI's own host code with the kernels replaced by tags and the launch call by a record)."""
import csv
import itertools
import math
import os
import subprocess
from pathlib import Path

import pytest

import test_gpu_backward
import test_gpu_parity

ROOT = Path(__file__).resolve().parent.parent
ROCM = Path(os.environ.get("ROCM_PATH", "/opt/rocm"))
HIPCC = ROCM / "bin" / "hipcc"
CLANG = ROCM / "llvm" / "bin" / "clang++"
pytestmark = pytest.mark.skipif(not (HIPCC.exists() and CLANG.exists()), reason="ROCm compilers not available")

NORMS = {"softmax": 0, "sigmoid": 1, "relu": 2}
SPLITS = ("one_group", "two_groups", "four_groups")
OWN = (4, 4, 2)      # row (key) wavefronts per group and groups of each backward split
GROUPS = (1, 2, 4)


@pytest.fixture(scope="module")
def launches(tmp_path_factory):
    """launches([(kind, B, H, Hkv, S, D, attention()'s keywords, packed hint or 0), ...]): the
    answers of launch_shapes.cpp, split into words."""
    tmp = tmp_path_factory.mktemp("launch_shapes")
    inc = [f"-I{ROOT / 'include'}", f"-I{ROOT / 'chia_proj_amd' / 'csrc'}"]
    subprocess.run([str(HIPCC), "--offload-arch=gfx950", "-std=c++17", "-O1", "-fPIC", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", *inc, "-c", str(ROOT / "chia_proj_amd" / "csrc" / "attn_api.hip"),
                    "-o", str(tmp / "api.o")], check=True, capture_output=True)
    subprocess.run([str(CLANG), "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM / 'include'}", *inc,
                    str(ROOT / "tests" / "cpp" / "launch_shapes.cpp"), str(tmp / "api.o"), "-o", str(tmp / "exe"),
                    f"-L{ROCM / 'lib'}", "-lamdhip64", f"-Wl,-rpath,{ROCM / 'lib'}"], check=True)

    def run(calls):
        text = "".join(
            f"{kind} {NORMS[kw.get('norm', 'softmax')]} {B} {H} {Hkv} {S} {D} {int(kw.get('causal', True))} "
            f"{kw.get('window', 0)} {kw.get('dilation', 1)} {kw.get('block', 0)} {kw.get('prefix', 0)} "
            f"{kw.get('softcap', 0.0)} {int('alibi_slopes' in kw)} {int('head_scale' in kw)} {packed}\n"
            for kind, B, H, Hkv, S, D, kw, packed in calls)
        out = subprocess.run([str(tmp / "exe")], input=text, capture_output=True, text=True, check=True)
        answers = [line.split() for line in out.stdout.splitlines()]
        assert len(answers) == len(calls)
        return answers

    return run


def _rows(S, kw):
    """Tokens of the first (longest) dilation residue, and the number of residues."""
    dil = min(kw.get("dilation", 1), S)
    return -(-S // dil), dil


def test_group_cases_run_the_shapes_they_name(launches):
    """The GPU tests of the workgroup shapes (test_key_groups, test_backward_query_groups,
    test_backward_key_groups): the launch rule takes the shape in each case's name."""
    fwd = test_gpu_parity.KEY_GROUPS
    for case, got in zip(fwd, launches([("fwd", B, H, H, S, D, kw, 0) for _, B, H, S, D, kw in fwd])):
        assert case[0].split("_")[0] == got[0], (case, got)
    dkdv = test_gpu_backward.SPLIT
    for case, got in zip(dkdv, launches([("bwd", *c[1:], 0) for c in dkdv])):
        assert case[0].startswith(SPLITS[int(got[3])]), (case, got)
        assert int(got[6]) == int("head_scale" in case[-1] and case[2] > case[3]), (case, got)
    dq = test_gpu_backward.DQ_SPLIT
    for case, got in zip(dq, launches([("bwd", B, H, H, S, D, kw, 0) for _, B, H, S, D, kw in dq])):
        assert case[0].startswith(SPLITS[int(got[0])]), (case, got)


def test_adversarial_cases_run_the_cores_they_mean(launches):
    """The shapes of test_softmax_rising_scores and test_alibi_softmax_tile_order at head dim 64."""
    def core(shape, S, **kw):
        B, H = shape
        return launches([("fwd", B, H, H, S, 64, kw, 0)])[0][0]

    B, H, S = test_gpu_parity.PAIRED_CAUSAL
    for kw in (dict(), dict(alibi_slopes=1), dict(head_scale=1)):
        assert core((B, H), S, causal=True, **kw) == "paired"
        assert core((4, 16), 2048, causal=False, **kw) == "paired"
        assert core((4, 16), 2048, causal=True, **kw) == "one"
        assert core((1, 2), 512, causal=True, **kw) == core((1, 2), 700, causal=False, **kw) == "keys4"
    assert core((B, H), S, causal=True, softcap=50.0) == "one"
    for mask in (dict(causal=True, prefix=256), dict(causal=True, window=256), dict(causal=False, block=256)):
        assert core((4, 16), 2048, **mask) == "one"
        assert core((1, 2), 512, **mask) == ("one" if "block" in mask else "keys4")


MASKS = [dict(causal=True), dict(causal=False), dict(causal=True, window=256), dict(causal=False, window=300),
         dict(causal=True, block=200), dict(causal=True, dilation=3), dict(causal=True, prefix=256)]
SCORES = [dict(), dict(alibi_slopes=1), dict(softcap=30.0), dict(softcap=80.0)]


def test_grids_cover_every_block(launches):
    """Every call of a sweep (masks, normalisers, score modifiers, packed batches with and
    without the hint) launches kernels that exist, on a grid with a workgroup for every block
    of rows (keys) of every slice; the fixed reference only for softcap softmax with a cap up
    to 54, and at head dim 64 not on full rows or packed causal ones."""
    calls = []
    for B, H, S, D in itertools.product((1, 4), (2, 16), (1, 64, 129, 777, 2048, 4097), (64, 128)):
        for mask, norm, score in itertools.product(MASKS, NORMS, SCORES):
            kw = dict(mask, norm=norm, **score)
            for packed in (0, 8 * (B * S // 16 + 1), 10 ** 9):
                for Hkv in (H, H // 2):
                    calls += [(kind, B, H, Hkv, S, D, kw, packed) for kind in ("fwd", "bwd")]
    seen = set()
    for (kind, B, H, Hkv, S, D, kw, packed), got in zip(calls, launches(calls)):
        case = (kind, B, H, Hkv, S, D, kw, packed, got)
        rows, residues = _rows(S, kw)
        slices, blocks = B * H * residues, -(-rows // 128)
        if kind == "fwd":
            core, threads, grid, fixed = got[0], *map(int, got[1:])
            pairs = slices * -(-blocks // 2)
            want = {"paired": (256, {pairs}), "zigzag2": (512, {pairs}), "keys2": (512, {slices * blocks}),
                    "keys4": (512, {slices * -(-rows // 64)}),
                    "one": (256, {slices * blocks, pairs} if D == 128 else {slices * blocks})}[core]
            assert threads == want[0] and grid in want[1], case
            assert core != "zigzag2" or D == 128, case
            full = not kw["causal"] and "window" not in kw
            if fixed:
                assert kw["norm"] == "softmax" and kw.get("softcap") == 30.0, case
                plain = not any(m in kw for m in ("window", "block", "prefix"))
                assert D == 128 or not (full or (packed and plain)), case
            seen.add((core, D, fixed))
        else:
            for at, (heads, per) in ((0, (H, "q")), (3, (Hkv, "kv"))):
                split, threads, grid = map(int, got[at:at + 3])
                assert threads == 64 * OWN[split] * GROUPS[split], case
                assert grid == B * heads * residues * -(-rows // (32 * OWN[split])), case
                seen.add((per, D, split))
    assert {(c, D, 0) for c in ("one", "keys2", "keys4", "paired") for D in (64, 128)} <= seen
    assert {(per, D, s) for per in ("q", "kv") for D in (64, 128) for s in range(3)} <= seen


def test_benchmark_shapes_launch_the_nominal_schedule(launches):
    """The headline and north-star suites launch the schedule whose tile counts the FLOP
    accounting quotes; a small grid need not."""
    from chia_proj_amd import plan
    from chia_proj_amd.accounting import core_plan_kwargs
    from chia_proj_amd.workloads import headline_suite, north_star_suite

    cases, plans, calls = [], [], []
    for c in headline_suite() + north_star_suite():
        params = dict(c.params, temperature=[1.0] * c.H) if c.temperature else c.params
        kw = core_plan_kwargs(c.op, c.H, params)
        plans.append(plan(batch=c.B, heads=c.H, seqlen=c.S, head_dim=c.D, **kw))
        named = {k: kw[k] for k in ("norm", "causal", "window", "dilation", "block", "prefix", "softcap") if k in kw}
        named.update({k: 1 for k, on in (("alibi_slopes", kw["alibi"]), ("head_scale", kw["head_scale"])) if on})
        cases.append(c.name)
        calls.append(("fwd", c.B, c.H, c.H, c.S, c.D, named, 0))
    for name, p, got in zip(cases, plans, launches(calls)):
        assert (got[0], int(got[1]), int(got[2])) == (
            "one" if p["block_n"] == 32 else "paired", 64 * p["waves"], p["workgroups"]), (name, p, got)
    small = plan(batch=1, heads=8, seqlen=512, head_dim=64, causal=True)
    assert small["waves"] == 2 and launches([("fwd", 1, 8, 8, 512, 64, dict(causal=True), 0)])[0][0] == "keys4"


# Measured times, us per call.  Forward: t0 one group, t1 keys2, t2 keys4, t3 the nominal schedule
# where it has a kernel.  Backward (dQ + dK/dV): t0-t2 dQ's splits, t3-t5 dK/dV's.
TIMES = ROOT / "profiles" / "launch_shape_times.csv"
MASK_OF = {"causal": dict(causal=True), "full": dict(causal=False), "window256": dict(causal=True, window=256),
           "local300": dict(causal=False, window=300), "block256": dict(causal=True, block=256),
           "dil2": dict(causal=True, dilation=2), "prefix": dict(causal=True, prefix=256)}


def test_rule_against_measured_times(launches):
    """The launch rule on the shapes timed with every workgroup shape: on average at most 3 %
    above the best one, and nowhere more than 6 % above one group per workgroup (forward: the
    nominal schedule), which runs without a rule."""
    rows = list(csv.DictReader(open(TIMES)))
    calls = []
    for r in rows:
        kw = dict(MASK_OF[r["mask"]], norm=r["norm"])
        if r["mod"]:
            kw.update(softcap=40.0) if r["mod"] == "softcap" else kw.update(alibi_slopes=1)
        calls.append((r["kind"], *(int(r[k]) for k in ("B", "H", "Hkv", "S", "D")), kw, 0))
    above, slower = {}, []
    for r, (kind, B, H, Hkv, S, D, kw, _), got in zip(rows, calls, launches(calls)):
        t = [float(r[f"t{i}"]) if r[f"t{i}"] else math.inf for i in range(6)]
        if kind == "fwd":
            n, residues = _rows(S, kw)
            pairs = B * H * residues * -(-(-(-n // 128)) // 2)
            at = {"one": 0, "keys2": 1, "keys4": 2}.get(got[0], 3)
            if got[0] == "one" and n > 128 and int(got[2]) == pairs:
                at = 3  # pairs of blocks, one group
            picks = [("fwd", t[at], min(t[:4]), t[3] if t[3] < math.inf else t[0])]
        else:
            picks = [("dq", t[int(got[0])], min(t[:3]), t[0]), ("dkdv", t[3 + int(got[3])], min(t[3:]), t[3])]
        for name, pick, best, before in picks:
            above.setdefault((name, D), []).append(math.log(pick / best))
            if pick > 1.06 * before:
                slower.append((r, name, got))
    assert not slower, slower
    for key, logs in above.items():
        mean = math.exp(sum(logs) / len(logs))
        print(key, len(logs), f"{mean:.4f}")
        assert mean <= 1.03, (key, mean)
