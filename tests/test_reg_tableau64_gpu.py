"""The FP64 optimality LP with its tableau in registers: every record and basis
equals the oracle's at the edges of the register shapes (rows per workgroup,
rows held in LDS, column slots, columns past the slots), where options end its
loops early, for cold starts with several lambda swaps, and as the re-solve of
a mixed-precision call."""
import os

import numpy as np
import pytest

from conftest import ROOT
from mpqpcudasolver_amd import assemble_lps, load_library, synthetic_mpqp
from oracle_lib import OracleLib
from parity import compare_runs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def libs():
    hip = load_library()
    assert hip.warm_up() == 0, hip.last_error()
    return hip, OracleLib(os.path.join(ROOT, "oracle", "_build", "libmpqp_oracle.so"))


def _pair(libs, lp, k, precision=0, **opts):
    hip, orc = libs
    hip.set_options(record=2, precision=precision, **opts)
    g = hip.run(lp, k_max=k, records=True, bases=True)
    st = hip.stats()
    hip.set_options()
    orc.set_options(record=2, precision=precision, **opts)
    o = orc.run(lp, k_max=k, records=True, bases=True)
    orc.set_options()
    return g, o, st


# (n, m, p, rows M2, columns K2, in registers): the last row or column of a
# register shape and the first past it, one row, rows in LDS, the first shape
# that stays split between LDS and global memory
SHAPES = [(2, 6, 1, 17, 11, True), (5, 19, 2, 48, 28, True), (4, 20, 2, 49, 28, True), (9, 33, 2, 80, 46, True),
          (45, 15, 2, 80, 64, True), (46, 15, 2, 81, 65, True), (13, 55, 2, 128, 72, True), (14, 55, 2, 129, 73, True),
          (77, 45, 4, 176, 128, True), (28, 70, 4, 177, 104, True), (78, 45, 4, 177, 129, True),
          (13, 117, 4, 256, 136, True), (14, 117, 4, 257, 137, True), (53, 129, 12, 336, 196, True),
          (54, 129, 12, 337, 197, False)]


@pytest.mark.parametrize("n,m,p,rows,cols,held", SHAPES, ids=[f"{s[3]}x{s[4]}" for s in SHAPES])
@pytest.mark.parametrize("batching", [0, 1])
def test_register_shapes(libs, n, m, p, rows, cols, held, batching):
    print(f"case: FP64 register tableau n={n} m={m} p={p}, |S| <= 1, batching {batching}", flush=True)
    lp = assemble_lps(synthetic_mpqp(n, m, p, 5))
    assert (lp.M2, lp.K2) == (rows, cols)
    g, o, st = _pair(libs, lp, 1, batching=batching)
    assert (st["split_rows_fp64"] == lp.M2) == held
    assert compare_runs(g, o) == []


ENDS = [("p1_iter_cap", dict(max_iter_phase1=3)), ("p1_stall", dict(stall_exit=2)), ("p2_iter_cap", dict(max_iter_phase2=1)),
        ("no_perturb_delay", dict(stall_perturb=0)), ("p1_unbounded", dict(tol_minus=-10.0)), ("singular", dict(licq_tol=0.3)),
        ("cold", dict(warm_start=0))]


@pytest.mark.parametrize("name,opts", ENDS, ids=[e[0] for e in ENDS])
def test_register_loop_ends(libs, name, opts):
    print(f"case: FP64 register tableau n=8 m=24 p=3 |S| <= 3, {name} {opts}", flush=True)
    lp = assemble_lps(synthetic_mpqp(8, 24, 3, 11))
    g, o, _ = _pair(libs, lp, 3, **opts)
    assert compare_runs(g, o) == []


def test_cold_starts_with_rows_in_lds(libs):
    print("case: FP64 register tableau with rows in LDS, cold starts n=100 m=40 p=4 |S| <= 2", flush=True)
    lp = assemble_lps(synthetic_mpqp(100, 40, 4, 3))
    g, o, st = _pair(libs, lp, 2, warm_start=0)
    assert st["split_rows_fp64"] == lp.M2
    assert compare_runs(g, o) == []


def test_fp64_resolve_of_a_mixed_call(libs):
    """Every candidate fails certification (tolerance 0) and is solved again."""
    print("case: FP64 register re-solve n=8 m=24 p=3 |S| <= 2", flush=True)
    lp = assemble_lps(synthetic_mpqp(8, 24, 3, 11))
    g, o, _ = _pair(libs, lp, 2, precision=1, certify_tol=1e-300, restart_pct=100)
    assert int(g.records["repivots"].sum()) > 0
    assert np.array_equal(g.records["repivots"], o.records["repivots"])
    assert compare_runs(g, o) == []
