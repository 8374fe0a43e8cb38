"""The driver's use of runs of iterations (tea_engine_cg_run, _ppcg_run,
_cheby_run), over the oracle with a library in front of it that answers the
runs otherwise (CPU)."""
from __future__ import annotations

import subprocess

import pytest

from tealeaf_cuda_amd import TeaError, run_deck

from test_gpu_configs import _same
from test_gpu_parity import DECKS, _deck

# A library that has its own run entry points and the oracle's everything else.
FRONT = r"""
#include <dlfcn.h>
#include <stdlib.h>
#include <string.h>

void tea_engine_cg_begin_ur(int, double, double, double *, double *);

static int refused(const char *name)     /* TEA_TEST_RUNS=<n>: the runs after the first n are refused */
{
    static int runs;
    const char *n = getenv(name);
    return n && runs++ >= atoi(n);
}

int tea_engine_cg_run(int with_p, double beta, double rro, int max_its, const double *stop, double *pw, double *rrn)
{
    int (*run)(int, double, double, int, const double *, double *, double *) = dlsym(RTLD_NEXT, "tea_engine_cg_run");
    double s[9];
    if (refused("TEA_TEST_RUNS")) return 0;
    memcpy(s, stop, sizeof s);
    if (getenv("TEA_TEST_BLIND")) s[3] = 0.0;     /* goes past the replacements */
    return run(with_p, beta, rro, max_its, s, pw, rrn);
}

int tea_engine_ppcg_run(int from_inner, int with_p, double beta, double rro, double theta, int inner_steps,
                        int max_its, const double *stop, double *values, int *at_ur, double *rrn_end)
{
    int (*run)(int, int, double, double, double, int, int, const double *, double *, int *, double *) =
        dlsym(RTLD_NEXT, "tea_engine_ppcg_run");
    if (refused("TEA_TEST_RUNS")) return 0;
    return run(from_inner, with_p, beta, rro, theta, inner_steps, max_its, stop, values, at_ur, rrn_end);
}

int tea_engine_cheby_run(int step, int n, int check_from, double error, double target, int max_its, double *rr)
{
    int (*run)(int, int, int, double, double, int, double *) = dlsym(RTLD_NEXT, "tea_engine_cheby_run");
    if (refused("TEA_TEST_RUNS")) return 0;
    return run(step, n, check_from, error, target, max_its, rr);
}
"""


@pytest.fixture
def front(oracle_so, oracle_env, driver_built, tmp_path):
    oracle_env("dot2")
    src, so = tmp_path / "front.c", tmp_path / "libfront.so"
    src.write_text("#define _GNU_SOURCE\n" + FRONT)
    subprocess.run(["gcc", "-O1", "-w", "-fPIC", "-shared", "-o", str(so), str(src), "-Wl,--no-as-needed",
                    str(oracle_so), f"-Wl,-rpath,{oracle_so.parent}", "-ldl"], check=True)
    return so


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_cg_run_past_a_replacement_is_an_error(precision, front, monkeypatch, tmp_path):
    kw = dict(DECKS["mixed_cg_block"], inner_precision=precision)
    path = _deck(**kw).write(tmp_path / "tea.in")
    assert sum(run_deck(path, backend=front).refinements) > 3      # replacements inside the solves
    monkeypatch.setenv("TEA_TEST_BLIND", "1")
    with pytest.raises(TeaError, match="went past a residual replacement"):
        run_deck(path, backend=front)


RUN_DECKS = {name: DECKS[name] for name in ("cg_block", "cheby_diag", "ppcg_diag_h2", "mixed_ppcg_block",
                                            "mixed_cg_block", "mixed_restart_ppcg_block", "refined_fp64_ppcg_block",
                                            "mixed_cheby_block")}
RUN_DECKS["refined_fp64_ppcg_diag"] = dict(DECKS["refined_fp64_ppcg_block"], preconditioner="jac_diag",
                                           reliable_delta=0.05)
RUN_DECKS["mixed_ppcg_none"] = dict(DECKS["mixed_ppcg_block"], preconditioner="none", reliable_delta=0.05)
# stopped by tl_max_iters inside and between replacements
for its in (25, 26, 27, 28):
    RUN_DECKS[f"mixed_ppcg_block_{its}"] = dict(DECKS["mixed_ppcg_block"], reliable_delta=0.3, max_iters=its)


@pytest.mark.parametrize("runs", [0, 1, 2, 3, 5])
@pytest.mark.parametrize("name", sorted(RUN_DECKS))
def test_runs_refused_in_mid_solve(name, runs, front, oracle_so, monkeypatch, tmp_path):
    """From any run on, the single calls take over: the same results."""
    path = _deck(**RUN_DECKS[name]).write(tmp_path / "tea.in")
    want = run_deck(path, backend=oracle_so)
    monkeypatch.setenv("TEA_TEST_RUNS", str(runs))
    _same(run_deck(path, backend=front), want)
