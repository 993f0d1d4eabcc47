"""The FP32 optimality LP with its tableau in registers: every record and
basis equals the oracle's at the edges of the register shapes (rows per
workgroup, column slots, columns past the slots), and where options end its
loops early."""
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


def _pair(libs, lp, k, **opts):
    hip, orc = libs
    hip.set_options(record=2, precision=1, **opts)
    g = hip.run(lp, k_max=k, records=True, bases=True)
    st = hip.stats()
    hip.set_options()
    orc.set_options(record=2, precision=1, **opts)
    o = orc.run(lp, k_max=k, records=True, bases=True)
    orc.set_options()
    return g, o, st


# (n, m, p, rows M2, columns K2): the last row or column of a register shape
# and the first past it, a single column slot, whole slots without extra columns
SHAPES = [(5, 12, 2, 34, 21), (20, 40, 2, 105, 64), (20, 41, 2, 107, 65), (27, 70, 4, 176, 103), (28, 70, 4, 177, 104),
          (77, 45, 4, 176, 128), (60, 118, 12, 321, 192), (60, 122, 12, 329, 196), (61, 122, 12, 330, 197),
          (61, 133, 12, 352, 208)]


@pytest.mark.parametrize("n,m,p,rows,cols", SHAPES, ids=[f"{s[3]}x{s[4]}" for s in SHAPES])
def test_register_shapes(libs, n, m, p, rows, cols):
    print(f"case: register tableau n={n} m={m} p={p}, |S| <= 1", flush=True)
    lp = assemble_lps(synthetic_mpqp(n, m, p, 5))
    assert (lp.M2, lp.K2) == (rows, cols)
    g, o, st = _pair(libs, lp, 1)
    assert not st["tableau_global"] & 2 and st["split_rows_fp32"] == lp.M2
    assert compare_runs(g, o) == []


ENDS = [("p1_iter_cap", dict(max_iter_phase1=3)), ("p1_stall", dict(stall_exit=2)), ("p2_iter_cap", dict(max_iter_phase2=1)),
        ("no_perturb_delay", dict(stall_perturb=0)), ("p1_unbounded", dict(tol32=10.0)), ("singular", dict(licq32=0.3)),
        ("cold", dict(warm_start=0)), ("late_restart", dict(restart_pct=100))]


@pytest.mark.parametrize("name,opts", ENDS, ids=[e[0] for e in ENDS])
def test_register_loop_ends(libs, name, opts):
    print(f"case: register tableau n=8 m=24 p=3 |S| <= 3, {name} {opts}", flush=True)
    lp = assemble_lps(synthetic_mpqp(8, 24, 3, 11))
    g, o, _ = _pair(libs, lp, 3, **{"restart_pct": 100, **opts})
    assert compare_runs(g, o) == []
    assert np.array_equal(g.records["repivots"], o.records["repivots"])


# ------------------------------------------------------------ the root tableau

def _with_w_entry(lp):
    """The LP with one off-diagonal entry in the block of the w pivots."""
    lp.A2 = lp.A2.copy(order="F")
    lp.A2[lp.M2 - lp.n_c + 3, lp.n_x + lp.n_t + 1] = 0.25
    return lp


ROOTS = [("columns", lambda lp: lp, {}), ("w_block_not_diagonal", _with_w_entry, {}),
         ("w_pivots_unusable", lambda lp: lp, dict(licq_tol=2.0))]


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("name,change,opts", ROOTS, ids=[r[0] for r in ROOTS])
def test_root_paths(libs, name, change, opts, precision):
    """The root built column by column, and by the general elimination where
    the w block is not diagonal (or has no usable pivot): records and bases
    equal the oracle's."""
    print(f"case: root tableau, {name}, precision {precision}", flush=True)
    hip, orc = libs
    lp = change(assemble_lps(synthetic_mpqp(7, 20, 3, 4)))
    runs = []
    for lib in (hip, orc):
        lib.set_options(record=2, precision=precision, **opts)
        runs.append(lib.run(lp, k_max=2, records=True, bases=True))
        lib.set_options()
    assert compare_runs(*runs) == []
    if name == "w_pivots_unusable":
        assert np.all(runs[0].records["p1_status"][runs[0].records["feasible"] == 1] == 5)
