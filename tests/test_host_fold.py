"""Argument checks of the folding entry points that return before any
device work (CPU): parameter ranges, the length limit, the pipeline's
minimum of two sequences, the locarna_rnafold_pp program's refusals, and the
workgroups and LDS that a launch is planned with (lcg_fold_plan)."""
import os
import subprocess

import pytest

from locarna_amd import api


@pytest.mark.parametrize("kw", [dict(min_prob=-0.1), dict(min_prob=1.0), dict(max_bp_span=0),
                                dict(max_bp_span=-2)])
def test_fold_parameter_ranges(kw):
    with pytest.raises(api.LcgError, match="fold parameters"):
        api.Fold(["ACGUACGUACGU"], **kw)


def test_fold_length_limit():
    with pytest.raises(api.LcgError, match="folding limit of 4096"):
        api.Fold(["ACGU" * 1024 + "A"])


def test_mlocarna_needs_two_sequences():
    with pytest.raises(api.LcgError):
        api.Mlocarna(["a"], ["ACGUACGUACGU"])


@pytest.mark.parametrize("args,stdin,msg", [(["--noLP"], "x ACGU\n", "not supported"),
                                            (["--in-loop"], "x ACGU\n", "not supported"),
                                            ([], ">a\nACGU\n>b\nACGU\n", "more than one sequence"),
                                            (["--bogus"], "x ACGU\n", "unknown option")])
def test_rnafold_pp_refusals(args, stdin, msg):
    exe = os.path.join(os.path.dirname(api.__file__), "_build", "locarna_rnafold_pp")
    r = subprocess.run([exe] + args, input=stdin, text=True, capture_output=True, timeout=60)
    assert r.returncode != 0 and msg in r.stderr


@pytest.mark.parametrize("lens", [[75], [64, 128, 256], [300, 700], [65] * 130 + [3700], [65] * 130 + [129, 3602, 1200],
                                  [100] * 300 + [4096, 650], [200] * 255 + [257], [4096] * 5, [64] * 200 + [4096],
                                  [1, 4096] * 128, [52, 1, 30], [53, 20], [20] * 256, [20] * 257, [0]])
def test_plan_fits(lens):
    """Every sequence's part of the LDS is inside what the launch allocates, and
    workgroups that wait for each other are resident together."""
    plan, allocated = api.fold_plan(lens, 256)
    assert allocated <= 160 * 1024
    assert max(lds for _, _, lds in plan) <= allocated
    members = [k for k, _, _ in plan]
    assert min(members) >= 1 and (max(members) == 1 or sum(members) <= 256)
    assert all(c in (1, 2, 4) and (k == 1 or c == 1) for k, c, _ in plan) or {c for _, c, _ in plan} == {0}
    assert (max(lens) <= 52 and len(lens) <= 256) == (plan[0][1] == 0)
