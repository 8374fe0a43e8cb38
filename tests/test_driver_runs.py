"""The driver's use of runs of iterations (tea_engine_cg_run, _ppcg_run,
_cheby_run), over the oracle with a library in front of it that answers the
runs otherwise (CPU)."""
from __future__ import annotations

import subprocess

import pytest

from tealeaf_cuda_amd import TeaError, run_deck

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
