"""Runs of solver iterations in one launch (tea_engine_cg_run, _ppcg_run,
_cheby_run) against the oracle's composition of the single calls, bit for bit:
the values returned and every field afterwards.

Sizes: one workgroup, bands one column short of, at and beyond the 62 a band
owns, last strips of one to four rows, fewer strips than waves, tiles of
several strips per wave up to the most that fits (a mesh of one row of tiles,
whose height sets the strips), and a mesh one band too wide for the chip, which
is refused and left as it was.
"""
from __future__ import annotations

import numpy as np
import pytest

from tealeaf_cuda_amd import Deck, Engine, run_deck
from tealeaf_cuda_amd import runtime as rt

from test_gpu_parity import DECKS, _deck, _prepare, _randomise, _randomise32

pytestmark = pytest.mark.gpu

NEVER = [-1.0, 1e9, -1.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0]
STOPS = {
    "never": NEVER,
    "error": [1e300] + NEVER[1:],
    "switch": [-1.0, 3.0, 1e300] + NEVER[3:],
    "replacement_first_q": NEVER[:3] + [1.0, 0.0, 0.0, 1.0, 1e200, 0.0],
    "replacement_given_q": NEVER[:3] + [1.0, 1.0, 1e-200, 1.0, 1e-3, 1e300],
    "replacement_not_due": NEVER[:3] + [1.0, 0.0, 0.0, 1.0, 1e-300, 0.0],
}
ALPHAS = [0.3, 0.5, 0.7, 0.2, 0.6, 0.4, 0.35, 0.55, 0.25, 0.45, 0.3, 0.5]
BETAS = [1.1, 0.9, 0.8, 1.2, 0.7, 1.0, 0.95, 0.85, 1.05, 0.75, 0.9, 1.1]
RUNS = {
    "cg": [("never", lambda e, s: e.cg_run(True, 0.61, 0.8, 5, s)),
           ("never", lambda e, s: e.cg_run(False, 0.0, 0.8, 1, s)),
           ("error", lambda e, s: e.cg_run(True, 0.61, 0.8, 5, s)),
           ("switch", lambda e, s: e.cg_run(True, 0.61, 0.8, 5, s)),
           ("replacement_first_q", lambda e, s: e.cg_run(False, 0.0, 0.8, 5, s)),
           ("replacement_given_q", lambda e, s: e.cg_run(True, 0.61, 0.8, 5, s)),
           ("replacement_not_due", lambda e, s: e.cg_run(True, 0.61, 0.8, 4, s)),
           # two runs, the second from what the first leaves owed; then the single call, then a norm
           ("never", lambda e, s: (e.cg_run(True, 0.61, 0.8, 2, s), e.cg_run(True, 0.3, 1.1, 2, s),
                                   e.cg_begin_ur(True, 0.2, 0.9), e.calc_2norm(2)))],
    "ppcg": [("never", lambda e, s: e.ppcg_run(False, True, 0.45, 0.8, 1.7, 5, 3, s)),
             ("never", lambda e, s: e.ppcg_run(False, False, 0.0, 0.8, 1.7, 1, 1, s)),
             ("never", lambda e, s: e.ppcg_run(True, False, 0.0, 0.8, 1.7, 4, 2, s)),
             ("error", lambda e, s: e.ppcg_run(False, True, 0.45, 0.8, 1.7, 3, 3, s)),
             ("replacement_first_q", lambda e, s: e.ppcg_run(False, True, 0.45, 0.8, 1.7, 3, 3, s)),
             ("replacement_given_q", lambda e, s: e.ppcg_run(True, True, 0.45, 0.8, 1.7, 3, 3, s)),
             ("never", lambda e, s: (e.ppcg_iteration(False, 0.0, 1.7, 10),
                                     e.ppcg_run(False, True, 0.45, 0.8, 1.7, 10, 2, s),
                                     e.ppcg_iteration(True, 0.3, 1.7, 10), e.calc_2norm(1)))],
    "chebyshev": [("never", lambda e, s: (e.cheby_init(ALPHAS, BETAS, 1.3), e.cheby_run(1, 1, 10**6, 1.0, 0.0, 7))),
                  ("never", lambda e, s: (e.cheby_init(ALPHAS, BETAS, 1.3), e.cheby_run(1, 7, 8, 2.0, 0.0, 9),
                                          e.calc_2norm(1), e.cheby_run(10, 16, 8, 2.0, 0.0, 1), e.cheby_iterate(11))),
                  ("never", lambda e, s: (e.cheby_init(ALPHAS, BETAS, 1.3), e.cheby_iterate(1),
                                          e.cheby_run(2, 2, 5, 1.0, 1e300, 6)))],
}
SMALL = [(3, 2), (61, 5), (62, 33), (63, 34), (125, 71), (250, 131)]


def _check(g, c, solver, prec, bits, nx, ny, runs, tmp_path):
    for k, (stop, fn) in enumerate(runs):
        print(f"[gpu resident] {solver}/{prec} fp{bits} {nx}x{ny} run {k} ({stop})", flush=True)
        outs = []
        for e in (g, c):
            _prepare(e, tmp_path, solver, prec, nx=nx, ny=ny, halo=2)
            if bits == 32:
                e.set_precision(32)
                e.mp_setup()
        rand = _randomise if bits == 64 else _randomise32
        rand((g, c), seed=k)
        for e in (g, c):
            e.cg_init()
            if solver == "ppcg":
                e.ppcg_init_constants(ALPHAS, BETAS)
        rand((g, c), seed=100 + k)
        outs = [repr(fn(e, STOPS[stop])) for e in (g, c)]   # (by text: random fields may overflow to nan)
        assert outs[0] == outs[1], k
        for fid in range(1, 20):
            if bits == 32 and fid in (rt.XFIELD_CP, rt.XFIELD_BFP):
                continue
            a, b = (e.get_field(fid) if bits == 64 else e.get_field32(fid) for e in (g, c))
            assert np.array_equal(a, b, equal_nan=True), f"run {k}: field {fid}"


@pytest.mark.parametrize("bits", [64, 32])
@pytest.mark.parametrize("prec", ["none", "jac_diag", "jac_block"])
@pytest.mark.parametrize("solver", ["cg", "ppcg", "chebyshev"])
def test_runs_bitwise(solver, prec, bits, oracle_so, oracle_env, tmp_path):
    oracle_env("dot2")
    g, c = Engine(), Engine(oracle_so)
    try:
        for nx, ny in SMALL:
            _check(g, c, solver, prec, bits, nx, ny, RUNS[solver], tmp_path)
    finally:
        g.finalize()
        c.finalize()


# one row of tiles: ny / 4 strips in 8 waves
@pytest.mark.parametrize("bits,ny", [(64, 34), (64, 65), (64, 97), (64, 127), (32, 129), (32, 161), (32, 254)])
@pytest.mark.parametrize("solver,prec", [("cg", "none"), ("cg", "jac_block"), ("ppcg", "jac_diag"),
                                         ("ppcg", "jac_block"), ("chebyshev", "jac_block")])
def test_runs_bitwise_tall_tiles(solver, prec, bits, ny, oracle_so, oracle_env, tmp_path):
    oracle_env("dot2")
    g, c = Engine(), Engine(oracle_so)
    try:
        _check(g, c, solver, prec, bits, 62 * 129 + 1, ny, RUNS[solver][:1], tmp_path)
    finally:
        g.finalize()
        c.finalize()


# several rows of tiles with several strips per wave (p, u, r and rstore of PPCG then stay in memory), the last row
# of tiles and the last strip short; the second run of a solve; fewer inner steps than strips per wave
MORE_PPCG = [("never", lambda e, s: (e.ppcg_run(False, False, 0.0, 0.8, 1.7, 3, 2, s),
                                     e.ppcg_run(False, True, 0.45, 0.8, 1.7, 3, 2, s))),
             ("never", lambda e, s: e.ppcg_run(False, True, 0.45, 0.8, 1.7, 1, 3, s))]


@pytest.mark.parametrize("bits,nx,ny", [(64, 1235, 390), (32, 1235, 775)])      # 2 and 3 strips
@pytest.mark.parametrize("solver,prec", [("ppcg", "none"), ("ppcg", "jac_diag"), ("ppcg", "jac_block"),
                                         ("cg", "jac_diag"), ("cg", "jac_block"), ("chebyshev", "none")])
def test_runs_bitwise_on_a_grid_of_tiles(solver, prec, bits, nx, ny, oracle_so, oracle_env, tmp_path):
    oracle_env("dot2")
    g, c = Engine(), Engine(oracle_so)
    try:
        runs = RUNS[solver] + (MORE_PPCG if solver == "ppcg" else [])
        _check(g, c, solver, prec, bits, nx, ny, runs, tmp_path)
    finally:
        g.finalize()
        c.finalize()


@pytest.mark.parametrize("bits,ny", [(64, 127), (32, 250)])                     # 4 and 8 strips
@pytest.mark.parametrize("prec", ["none", "jac_diag", "jac_block"])
def test_ppcg_runs_bitwise_with_the_most_strips(prec, bits, ny, oracle_so, oracle_env, tmp_path):
    oracle_env("dot2")
    g, c = Engine(), Engine(oracle_so)
    try:
        _check(g, c, "ppcg", prec, bits, 62 * 129 + 1, ny, [RUNS["ppcg"][5]] + MORE_PPCG, tmp_path)
    finally:
        g.finalize()
        c.finalize()


def test_mesh_too_wide_is_left_alone(tmp_path):
    g = Engine()
    try:
        _prepare(g, tmp_path, "cg", "none", nx=62 * 256 + 1, ny=3)
        g.cg_init()
        before = [g.get_field(fid) for fid in range(1, 20)]
        assert g.cg_run(True, 0.5, 1.0, 4, NEVER) == ([], [])
        for fid in range(1, 20):
            assert np.array_equal(before[fid - 1], g.get_field(fid), equal_nan=True)
    finally:
        g.finalize()


@pytest.mark.parametrize("name", sorted(DECKS))
def test_decks_without_runs(name, oracle_so, driver_built, oracle_env, monkeypatch, tmp_path):
    """TEA_RESIDENT=0: the separate kernels give the same results."""
    oracle_env("dot2")
    monkeypatch.setenv("TEA_RESIDENT", "0")
    print(f"[gpu resident] deck {name} without runs", flush=True)
    path = _deck(**DECKS[name]).write(tmp_path / "tea.in")
    gpu, cpu = run_deck(path), run_deck(path, backend=oracle_so)
    assert gpu.iterations == cpu.iterations and gpu.refinements == cpu.refinements
    assert gpu.ppcg_inner == cpu.ppcg_inner
    assert gpu.exact_error == cpu.exact_error
    for a, b in zip(gpu.summaries, cpu.summaries):
        assert a.values() == b.values(), (a, b)


# A run that does not start (part of the chip is taken: the workgroups' verdict is given from the host), after
# calls that leave fields owed, then the single calls: what they leave is what they leave without it.
NOT_STARTED = {
    "cg": [(lambda e: e.cg_begin_ur(True, 0.3, 0.9), lambda e: e.cg_run(True, 0.61, 0.8, 5, NEVER),
            lambda e: (e.cg_begin_ur(True, 0.61, 0.8), e.calc_2norm(2))),
           (lambda e: e.cg_begin_ur(True, 0.3, 0.9), lambda e: e.cg_run(True, 0.61, 0.8, 5, NEVER), lambda e: None)],
    "ppcg": [(lambda e: e.ppcg_iteration(True, 0.3, 1.7, 4),
              lambda e: e.ppcg_run(False, True, 0.45, 0.8, 1.7, 5, 3, NEVER),
              lambda e: (e.ppcg_iteration(True, 0.45, 1.7, 5), e.calc_2norm(1))),
             (lambda e: e.ppcg_iteration(True, 0.3, 1.7, 4),
              lambda e: e.ppcg_run(False, True, 0.45, 0.8, 1.7, 5, 3, NEVER), lambda e: None),
             (lambda e: e.ppcg_begin_ur(True, 0.3, 1.7), lambda e: e.ppcg_run(True, False, 0.0, 0.8, 1.7, 4, 2, NEVER),
              lambda e: (e.ppcg_inner_n(1, 4), e.ppcg_end(), e.calc_2norm(1))),
             (lambda e: e.ppcg_begin_ur(True, 0.3, 1.7), lambda e: e.ppcg_run(True, False, 0.0, 0.8, 1.7, 4, 2, NEVER),
              lambda e: None)],
    "chebyshev": [(lambda e: (e.cheby_init(ALPHAS, BETAS, 1.3), e.cheby_iterate_n(1, 3)),
                   lambda e: e.cheby_run(4, 4, 10**6, 1.0, 0.0, 5), lambda e: (e.cheby_iterate_n(4, 2), e.calc_2norm(1))),
                  (lambda e: (e.cheby_init(ALPHAS, BETAS, 1.3), e.cheby_iterate_n(1, 3)),
                   lambda e: e.cheby_run(4, 4, 10**6, 1.0, 0.0, 5), lambda e: None)],
}


@pytest.mark.parametrize("bits", [64, 32])
@pytest.mark.parametrize("prec", ["none", "jac_diag", "jac_block"])
@pytest.mark.parametrize("solver", sorted(NOT_STARTED))
def test_run_that_does_not_start(solver, prec, bits, oracle_so, oracle_env, monkeypatch, tmp_path, capfd):
    oracle_env("dot2")
    monkeypatch.setenv("TEA_RESIDENT_TAKEN", "0")
    g, c = Engine(), Engine(oracle_so)
    try:
        for k, (before, run, after) in enumerate(NOT_STARTED[solver]):
            print(f"[gpu resident] not started: {solver}/{prec} fp{bits}, {k}", flush=True)
            for e in (g, c):
                _prepare(e, tmp_path, solver, prec, nx=125, ny=71, halo=2)
                if bits == 32:
                    e.set_precision(32)
                    e.mp_setup()
            rand = _randomise if bits == 64 else _randomise32
            rand((g, c), seed=k)
            for e in (g, c):
                e.cg_init()
                if solver == "ppcg":
                    e.ppcg_init_constants(ALPHAS, BETAS)
            rand((g, c), seed=100 + k)
            outs = []
            for e in (g, c):
                out = [before(e)]
                if e is g:
                    got = run(e)
                    assert not (got[0] if isinstance(got, tuple) else got)
                    assert "part of the GPU is taken" in capfd.readouterr().err
                out.append(after(e))
                outs.append(repr(out))
            assert outs[0] == outs[1], k
            for fid in range(1, 20):
                if bits == 32 and fid in (rt.XFIELD_CP, rt.XFIELD_BFP):
                    continue
                a, b = (e.get_field(fid) if bits == 64 else e.get_field32(fid) for e in (g, c))
                assert np.array_equal(a, b, equal_nan=True), f"case {k}: field {fid}"
    finally:
        g.finalize()
        c.finalize()


@pytest.mark.parametrize("runs", [0, 1, 2])
@pytest.mark.parametrize("name", ["cg_block", "cheby_diag", "ppcg_diag_h2", "mixed_cg_block", "mixed_ppcg_diag_h2",
                                  "refined_fp64_ppcg_block", "mixed_cheby_block"])
def test_decks_whose_runs_stop_starting(name, runs, oracle_so, driver_built, oracle_env, monkeypatch, tmp_path):
    oracle_env("dot2")
    monkeypatch.setenv("TEA_RESIDENT_TAKEN", str(runs))
    print(f"[gpu resident] deck {name}, {runs} runs start", flush=True)
    path = _deck(**DECKS[name]).write(tmp_path / "tea.in")
    gpu, cpu = run_deck(path), run_deck(path, backend=oracle_so)
    assert gpu.iterations == cpu.iterations and gpu.refinements == cpu.refinements
    assert gpu.ppcg_inner == cpu.ppcg_inner and gpu.exact_error == cpu.exact_error
    for a, b in zip(gpu.summaries, cpu.summaries):
        assert a.values() == b.values(), (a, b)
