"""Which kernel runs a call (MpqpStats.register_shapes), at both sides of every
register shape; and the kernels that a call reaches only by its options or by
unusual sizes, against the oracle: LDS tableaus (named workgroup sizes, many
parameter rows), split ones (plain, autotuned), and the register shapes with
columns by row, rows in LDS and several stage passes where options end their
loops early."""
import os

import numpy as np
import pytest

from conftest import ROOT
from mpqpcudasolver_amd import assemble_lps, load_library, synthetic_mpqp
from oracle_lib import OracleLib
from parity import compare_runs
from test_feas_registers_gpu import SHAPES as FEAS_SHAPES
from test_reg_tableau64_gpu import SHAPES as FP64_SHAPES
from test_reg_tableau_gpu import SHAPES as FP32_SHAPES

pytestmark = pytest.mark.gpu

# (rows, columns) of the kernels, smallest first
FP64 = [(48, 64), (80, 64), (128, 72), (176, 128), (256, 136), (336, 196)]
FP32 = [(88, 68), (128, 72), (176, 128), (256, 136), (352, 196), (352, 256)]
FEAS = [(128, 64), (160, 76), (160, 128)]


@pytest.fixture(scope="module")
def libs():
    hip = load_library()
    assert hip.warm_up() == 0, hip.last_error()
    return hip, OracleLib(os.path.join(ROOT, "oracle", "_build", "libmpqp_oracle.so"))


def _first(shapes, rows, cols):
    return next((i + 1 for i, (r, c) in enumerate(shapes) if rows <= r and cols <= c), 0)


def _shapes(stats):
    s = stats["register_shapes"]
    return {"fp64": s & 255, "fp32": s >> 8 & 255, "feas": s >> 16 & 255}


def _pair(libs, lp, k, **opts):
    hip, orc = libs
    hip.set_options(record=2, **opts)
    g = hip.run(lp, k_max=k, records=True, bases=True)
    st = hip.stats()
    hip.set_options()
    orc.set_options(record=2, **opts)
    o = orc.run(lp, k_max=k, records=True, bases=True)
    orc.set_options()
    return g, o, st


CHOICES = sorted({s[:3] for s in FP64_SHAPES + FP32_SHAPES + FEAS_SHAPES} | {(7, 15, 2), (8, 16, 2)})


@pytest.mark.parametrize("n,m,p", CHOICES)
@pytest.mark.parametrize("precision", [0, 1])
def test_chosen_shapes(libs, n, m, p, precision):
    print(f"case: kernel choice n={n} m={m} p={p}, precision {precision}", flush=True)
    hip = libs[0]
    lp = assemble_lps(synthetic_mpqp(n, m, p, 5))
    hip.set_options(precision=precision)
    hip.run(lp, k_max=0)
    st = hip.stats()
    hip.set_options()
    got = _shapes(st)
    feas = _first(FEAS, lp.M1, lp.K1) if (lp.M1 + 1) * (lp.K1 + 1) > 4800 else 0
    # the FP32 kernel is for tableaus of more than one wave's rows
    fp32 = _first(FP32, lp.M2, lp.K2) if precision == 1 and lp.M2 > 44 else 0
    if (fp32, lp.M2) == (2, 128):
        fp32 = 3  # half of its rows staged are more LDS than its six workgroups a CU have
    assert got == {"fp64": _first(FP64, lp.M2, lp.K2), "fp32": fp32, "feas": feas}


@pytest.mark.parametrize("batching", [0, 1])
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nt", [256, 512, 1024])
@pytest.mark.parametrize("nmp,k", [((8, 24, 3), 3), ((30, 62, 8), 1)])
def test_named_workgroup_sizes_use_lds(libs, nmp, k, nt, precision, batching):
    print(f"case: LDS tableau n,m,p={nmp} |S|<={k}, {nt} threads, precision {precision}, batching {batching}", flush=True)
    lp = assemble_lps(synthetic_mpqp(*nmp, 11))
    g, o, st = _pair(libs, lp, k, precision=precision, batching=batching, opt_threads=nt)
    assert _shapes(st) == {"fp64": 0, "fp32": 0, "feas": 0}
    # the 171 x 102 tableau fits in LDS in FP64 too
    assert st["tableau_global"] == 0
    assert compare_runs(g, o) == []


ENDS = [("p1_iter_cap", dict(max_iter_phase1=3)), ("p1_stall", dict(stall_exit=2)), ("p2_iter_cap", dict(max_iter_phase2=1)),
        ("no_perturb_delay", dict(stall_perturb=0)), ("p1_unbounded", dict(tol_minus=-10.0, tol32=10.0)),
        ("singular", dict(licq_tol=0.3, licq32=0.3)), ("cold", dict(warm_start=0))]


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("name,opts", ENDS, ids=[e[0] for e in ENDS])
def test_lds_loop_ends(libs, name, opts, precision):
    print(f"case: LDS tableau n=8 m=24 p=3 |S| <= 3, {name} {opts}, precision {precision}", flush=True)
    lp = assemble_lps(synthetic_mpqp(8, 24, 3, 11))
    g, o, st = _pair(libs, lp, 3, precision=precision, opt_threads=256, restart_pct=100, **opts)
    assert _shapes(st)["fp64"] == 0 and st["tableau_global"] == 0
    assert compare_runs(g, o) == []
    assert np.array_equal(g.records["repivots"], o.records["repivots"])


# columns by row; several slots, columns by row, rows in LDS (FP64), stage passes (FP32)
RICH = [((46, 15, 2), 2, 3, 1), ((53, 129, 12), 1, 6, 5)]


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nmp,k,shape64,shape32", RICH, ids=["extra_columns", "lds_rows"])
@pytest.mark.parametrize("name,opts", ENDS, ids=[e[0] for e in ENDS])
def test_register_loop_ends(libs, name, opts, nmp, k, shape64, shape32, precision):
    print(f"case: register tableau n,m,p={nmp} |S| <= {k}, {name} {opts}, precision {precision}", flush=True)
    lp = assemble_lps(synthetic_mpqp(*nmp, 11))
    g, o, st = _pair(libs, lp, k, precision=precision, restart_pct=100, **opts)
    assert _shapes(st)["fp64"] == shape64 and _shapes(st)["fp32"] == (shape32 if precision else 0)
    assert compare_runs(g, o) == []
    assert np.array_equal(g.records["repivots"], o.records["repivots"])


@pytest.mark.parametrize("batching", [0, 1])
@pytest.mark.parametrize("precision", [0, 1])
def test_lds_tableau_of_many_parameter_rows(libs, precision, batching):
    """More rows than any register shape, but few columns: an LDS tableau
    without any option, and the autotuner's choice of its workgroup size."""
    print(f"case: LDS tableau, 400 parameter rows, precision {precision}, batching {batching}", flush=True)
    prog = synthetic_mpqp(5, 12, 3, 7)
    rng = np.random.default_rng(2)
    rows = rng.standard_normal((400, 3))
    prog.A_t = np.vstack([prog.A_t, rows / np.linalg.norm(rows, axis=1, keepdims=True)])
    prog.b_t = np.vstack([prog.b_t.reshape(-1, 1), rng.uniform(0.5, 3.0, (400, 1))])
    lp = assemble_lps(prog)
    assert lp.M2 > 352
    for _ in range(2):
        g, o, st = _pair(libs, lp, 3, precision=precision, batching=batching)
        assert _shapes(st)["fp64"] == _shapes(st)["fp32"] == 0 and st["tableau_global"] == 0
        assert compare_runs(g, o) == []


# (n, m, p), options: a split tableau by request, and one larger than every register shape
SPLITS = [((60, 120, 12), dict(split_wgs=1)), ((60, 120, 12), dict(split_wgs=2)),
          ((62, 133, 12), dict()), ((62, 133, 12), dict(batching=1))]


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nmp,opts", SPLITS, ids=["1_plain", "2_plain", "large_plain", "large_autotuned"])
def test_split_tableaus(libs, nmp, opts, precision):
    print(f"case: split tableau n,m,p={nmp} |S| <= 1, {opts}, precision {precision}", flush=True)
    lp = assemble_lps(synthetic_mpqp(*nmp, 5))
    for _ in range(2):  # (the second call with the sizes that the autotuner has kept)
        g, o, st = _pair(libs, lp, 1, precision=precision, **opts)
        assert _shapes(st)["fp64"] == _shapes(st)["fp32"] == 0
        assert st["tableau_global"] & (2 if precision else 1)
        assert st["split_rows_fp32" if precision else "split_rows_fp64"] < lp.M2
        assert compare_runs(g, o) == []
