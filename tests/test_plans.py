"""The dispatcher's kernel choices, pinned on the CPU through the dry-run entry point
migemm_gemm_plan (validates and plans exactly as migemm_gemm_strided_batched_ex, launches
nothing, makes no HIP call): every BASELINE config, every caller shape of the path and the
regime table (tests/dispatch_cases.py). A change to the dispatcher shows up here as a
changed plan string; the GPU suite checks that real calls record the same plans
(tests/test_gemm_gpu.py::test_dry_run_plans_match_real_calls)."""
import random
import re

import pytest

import dispatch_cases as dc
from my_pytchon_opencl_lib_amd import _native


@pytest.fixture(autouse=True)
def auto_policy():
    prev = _native.set_gemm_policy(_native.MIGEMM_POLICY_AUTO)
    yield
    _native.set_gemm_policy(prev)


@pytest.mark.parametrize("name,spec,plan", dc.BASELINE + dc.CALLERS,
                         ids=[c[0] for c in dc.BASELINE + dc.CALLERS])
def test_plan_of_baseline_and_callers(name, spec, plan):
    assert _native.gemm_plan(*dc.args(**spec)) == plan


@pytest.mark.parametrize("name", dc.FP32)
def test_fp32_plan_behind_a_split_one(name):
    spec = next(s for n, s, _ in dc.BASELINE + dc.CALLERS if n == name)
    with _native.tuned(direct=2):
        assert _native.gemm_plan(*dc.args(**spec)) == dc.FP32[name]


@pytest.mark.parametrize("spec,plan", dc.AUTO_REGIMES)
def test_plan_of_regime_table(spec, plan):
    assert _native.gemm_plan(*dc.regime_args(spec)).startswith(plan)


def test_plan_validates_like_the_gemm_entry():
    a = dc.args(64, 64, 64)
    with pytest.raises(_native.MigemmArgumentError, match="sizes must be >= 1"):
        _native.gemm_plan(*dc.args(0, 64, 64))
    # C on top of A
    bad = list(a)
    bad[12] = bad[5]
    with pytest.raises(_native.MigemmArgumentError, match="overlaps"):
        _native.gemm_plan(*bad)
    with pytest.raises(_native.MigemmArgumentError, match="unknown flags"):
        _native.gemm_plan(*a[:-1], 2)


def test_plan_follows_policy_and_tuning():
    """The dry run sees the process-wide policy and tuning overrides as a real call does."""
    a = dc.args(4096, 4096, 4096)
    prev = _native.set_gemm_policy(_native.MIGEMM_POLICY_SMALL)
    try:
        assert _native.gemm_plan(*a).startswith("small ")
    finally:
        _native.set_gemm_policy(prev)
    with _native.tuned(tile=128, splitk=2):
        assert _native.gemm_plan(*a).startswith("tiled-direct tile=128x128 splits=2 ")
    with _native.tuned(direct=2):
        assert _native.gemm_plan(*a).startswith("tiled-direct tile=256x256 splits=1 ")
    assert _native.gemm_plan(*a).startswith("tiled-split tile=256x128 splits=1 ")


# (M, K, N, ta, tb, k ranges of the fp32 plan): products whose split plan has more ranges
PARTIALS = [(960, 4736, 704, 1, 0, 4), (1536, 4096, 3072, 0, 1, 2), (640, 1472, 1280, 0, 0, 4),
            (6400, 4096, 512, 0, 1, 3), (512, 6400, 4096, 1, 0, 1)]


@pytest.mark.parametrize("M,K,N,ta,tb,ranges", PARTIALS)
def test_partial_sums_fit_the_workspace_or_another_plan_runs(M, K, N, ta, tb, ranges):
    """With a workspace that holds the fp32 plan's partial sums but not the split plan's (a
    stream being captured) the fp32 plan runs in that workspace; with less, the call is
    refused. A launch of k ranges without a buffer for them is an error in any plan."""
    a = dc.args(M, N, K, ta=ta, tb=tb)
    fp32 = ranges * M * N * 4 if ranges > 1 else 0
    free = _native.gemm_plan(*a)
    for kib in (-(-fp32 // 1024) or 1, 1 << 20):
        with _native.tuned(plan_workspace=kib):
            plan = _native.gemm_plan(*a)
        if kib < 1 << 20:
            assert plan.startswith("tiled-direct ") and f"splits={ranges} " in plan
        else:
            assert plan == free and plan.startswith("tiled-split ")
    if ranges > 1:
        with _native.tuned(plan_workspace=fp32 // 1024 - 1):
            with pytest.raises(_native.MigemmRuntimeError, match="bytes of workspace are needed"):
                _native.gemm_plan(*a)


def test_split_plan_has_no_fewer_k_ranges_than_the_fp32_plan():
    """The error of a sum grows with the root of its k range: over products of 200-13000 the
    split kernel never runs fewer ranges than the fp32 plan it replaces."""
    rng = random.Random(3)
    splits = 0
    for _ in range(3000):
        M, K, N = (int(200 * 65 ** rng.random()) // 32 * 32 + rng.choice([0, 5]) for _ in range(3))
        a = dc.args(M, N, K, ta=rng.randrange(2), tb=rng.randrange(2))
        plan = _native.gemm_plan(*a)
        if plan.startswith("tiled-split "):
            splits += 1
            with _native.tuned(direct=2):
                fp32 = _native.gemm_plan(*a)
            ranges = [int(re.search(r"splits=(\d+) ", p)[1]) for p in (plan, fp32)]
            assert ranges[0] >= ranges[1], (plan, fp32)
    assert splits > 500


def test_no_plan_launches_k_ranges_without_a_buffer():
    """Products over the tiled family's range, each under workspaces of 1 KiB to 1 GiB: the
    dispatcher plans a launch or refuses for want of workspace, and what runs in a workspace
    runs in any larger one."""
    rng = random.Random(5)
    for _ in range(400):
        M, K, N = (rng.randrange(200, 6500) // 32 * 32 + rng.choice([0, 0, 1]) for _ in range(3))
        a = dc.args(M, N, K, ta=rng.randrange(2), tb=rng.randrange(2))
        ran = False
        for kib in [1 << e for e in range(0, 21, 2)]:
            with _native.tuned(plan_workspace=kib):
                try:
                    _native.gemm_plan(*a)
                    ran = True
                except _native.MigemmRuntimeError as e:
                    assert "bytes of workspace are needed" in str(e)
                    assert not ran, (M, K, N, a[:2], kib)
        assert ran, (M, K, N, a[:2])
