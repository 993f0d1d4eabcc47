"""The feasibility LP with its tableau in registers: every record and basis
equals the oracle's at the edges of its shapes (rows, column slots, columns
past the slots), on both sides of the size it starts at, and where options end
its loop early."""
import os

import pytest

from conftest import ROOT
from mpqpcudasolver_amd import assemble_lps, load_library, synthetic_mpqp
from oracle_lib import OracleLib
from parity import compare_runs

pytestmark = pytest.mark.gpu

# (n, m, p, rows M1, columns K1)
SHAPES = [(36, 76, 8, 92, 45), (40, 84, 8, 100, 49), (55, 120, 4, 128, 60), (59, 120, 4, 128, 64), (60, 120, 4, 128, 65),
          (55, 121, 4, 129, 60), (62, 136, 12, 160, 75), (63, 136, 12, 160, 76), (64, 136, 12, 160, 77),
          (62, 137, 12, 161, 75), (121, 40, 6, 52, 128), (122, 40, 6, 52, 129)]


def _pair(lp, k, **opts):
    hip, orc = load_library(), OracleLib(os.path.join(ROOT, "oracle", "_build", "libmpqp_oracle.so"))
    hip.set_options(record=2, **opts)
    g = hip.run(lp, k_max=k, records=True, bases=True)
    hip.set_options()
    orc.set_options(record=2, **opts)
    o = orc.run(lp, k_max=k, records=True, bases=True)
    orc.set_options()
    return g, o


@pytest.mark.parametrize("n,m,p,rows,cols", SHAPES, ids=[f"{s[3]}x{s[4]}" for s in SHAPES])
def test_feasibility_shapes(n, m, p, rows, cols):
    print(f"case: feasibility tableau n={n} m={m} p={p}, |S| <= 1", flush=True)
    lp = assemble_lps(synthetic_mpqp(n, m, p, 5))
    assert (lp.M1, lp.N1 - lp.M1) == (rows, cols)
    g, o = _pair(lp, 1)
    assert compare_runs(g, o) == []


ENDS = [("iter_cap", dict(max_iter_feas=1)), ("unbounded", dict(tol_plus=10.0)), ("cold", dict(warm_start=0)),
        ("no_screen", dict(licq_screen=0.0))]


@pytest.mark.parametrize("name,opts", ENDS, ids=[e[0] for e in ENDS])
def test_feasibility_ends(name, opts):
    print(f"case: feasibility tableau n=40 m=84 p=8 |S| <= 2, {name} {opts}", flush=True)
    lp = assemble_lps(synthetic_mpqp(40, 84, 8, 3))
    g, o = _pair(lp, 2 if name != "unbounded" else 1, **opts)
    assert compare_runs(g, o) == []
