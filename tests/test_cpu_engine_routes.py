"""The sanitised drivers run the host paths that the library has: every
launcher that the host sources call is defined in them, as it is in the
library, so none is chosen by whether it exists.  The chunks of iterations
that small CG solves run in one launch keep the solver's rules, and batched
PCG gives the same solution alone and in a batch on either side of the item
count above which an instance's sums are added up in launches of their own."""
import os
import shutil
import subprocess

import pytest

from conftest import PKG
from test_cpu_engine import ENG, batch_results, results  # noqa: F401  (the drivers' cases)


def _undefined_weak(path, *flags):
    out = subprocess.run(["nm", *flags, path], check=True, capture_output=True, text=True).stdout
    return [l.split()[-1] for l in out.splitlines() if l.split()[-2:-1] == ["w"] and "sipg" in l]


@pytest.mark.parametrize("driver", ["engine_driver", "batch_driver", "serve_driver"])
def test_no_launcher_is_optional_in_the_drivers(results, driver):  # noqa: F811  (builds them)
    if shutil.which("nm") is None:
        pytest.skip("no nm")
    assert _undefined_weak(os.path.join(ENG, "_build", driver)) == []


def test_no_launcher_is_optional_in_the_library():
    so = os.path.join(PKG, "lib", "libsipg_hip.so")
    if shutil.which("nm") is None or not os.path.exists(so):
        pytest.skip("no nm or library")
    assert _undefined_weak(so, "-D") == []


def test_small_plain_cg_is_the_reference_iteration(results):  # noqa: F811
    r = results["small_plain"]
    assert r["rc"] == 0 and r["chunks"] > 0 and r["iters"] == r["oracle_iters"] and r["diff"] <= 1e-11, r


def test_small_cg_iteration_cap(results):  # noqa: F811
    r = results["small_cap"]
    assert r["rc"] == 6 and r["chunks"] > 0 and r["iters"] == 37 and r["diff"] <= 1e-11, r


@pytest.mark.parametrize("case", ["small_replace", "small_noreplace", "small_near_floor"])
def test_small_cg_reaches_its_true_residual(results, case):  # noqa: F811
    # a replacement interrupts the chunks; the host polls at most two chunks
    # of 32 iterations behind
    r = results[case]
    tol = 1.5e-14 if case == "small_near_floor" else 1e-10
    assert r["rc"] == 0 and r["chunks"] > 0 and r["reps"] >= 1 and r["relres"] <= tol, r
    if case != "small_near_floor":
        assert r["oracle_iters"] <= r["iters"] <= r["oracle_iters"] + 64, r


def test_small_mixed_cycles(results):  # noqa: F811
    r = results["small_mixed"]
    assert r["rc"] == 0 and r["chunks"] > 0 and r["relres"] <= 1e-10 and r["diff"] <= 1e-8, r


def test_small_cg_breakdown(results):  # noqa: F811
    r = results["small_breakdown"]
    assert r["rc"] == 8 and r["chunks"] > 0, r


@pytest.mark.parametrize("case,tol", [("small_exact", 1e-6), ("small_exact_loose", 0.4), ("small_exact_p2", 1e-3)])
def test_small_cg_that_solves_exactly_is_no_breakdown(results, case, tol):  # noqa: F811
    # 4 and 9 unknowns: within a chunk the recursion falls to zero, or so low
    # that p.Ap does; the solve still finishes on its true residual
    r = results[case]
    assert r["rc"] == 0 and r["chunks"] > 0 and r["reps"] >= 1 and r["relres"] <= tol, r


def test_small_cg_does_not_run_past_its_tolerance_into_the_cap(results):  # noqa: F811
    # the reference iteration takes 177: a cap five above is enough for the
    # recursion and its final check
    r = results["small_near_cap"]
    assert r["oracle_iters"] == 177 and r["rc"] == 0 and r["chunks"] > 0 and r["iters"] <= 182, r


def test_batched_pcg_about_the_item_limit(batch_results):  # noqa: F811
    # 512, 9 (of degree 3), 513 and 525 items
    rows = batch_results["batch_items"]
    for r in rows:
        assert r["status"] == 0 and r["relres"] <= 1e-10 and r["reps"] >= 1 and r["alone_maxdiff"] == 0.0, r
    assert [r["totals"] > 0 for r in rows] == [False, False, True, True], rows
