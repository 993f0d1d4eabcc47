"""Candidate lists, children and final sets made on the device: a call without
records returns the oracle's active sets and counts over one block of
candidates and several, chunks around a block's 1024, and more final sets than
the counts' host buffer has rows for."""
import os

import pytest

from conftest import ROOT
from mpqpcudasolver_amd import assemble_lps, load_library, synthetic_mpqp
from oracle_lib import OracleLib

pytestmark = pytest.mark.gpu

CASES = [("k0", (10, 30, 8), 0, 0, 0), ("one_block", (12, 40, 10), 2, 0, 0), ("blocks", (10, 30, 8), 3, 0, 0),
         ("rows_past_buffer", (12, 40, 10), 3, 0, 0), ("chunk_1023", (10, 30, 8), 3, 0, 1023),
         ("chunk_1024", (10, 30, 8), 3, 0, 1024), ("chunk_1025", (10, 30, 8), 3, 2, 1025), ("chunk_31", (10, 30, 8), 2, 1, 31)]


@pytest.mark.parametrize("batching", [0, 1])
@pytest.mark.parametrize("name,nmp,k,k_min,chunk", CASES, ids=[c[0] for c in CASES])
def test_lists_match_oracle(name, nmp, k, k_min, chunk, batching):
    print(f"case: device lists {name} n,m,p={nmp} |S|<={k} k_min={k_min} max_chunk={chunk} batching={batching}", flush=True)
    lp = assemble_lps(synthetic_mpqp(*nmp, 5))
    hip, orc = load_library(), OracleLib(os.path.join(ROOT, "oracle", "_build", "libmpqp_oracle.so"))
    hip.set_options(record=0, batching=batching, max_chunk=chunk)
    g = hip.run(lp, k_max=k, k_min=k_min)
    st = hip.stats()
    hip.set_options()
    orc.set_options(record=1)
    o = orc.run(lp, k_max=k, k_min=k_min, records=True)
    orc.set_options()
    # chunks are visited depth first, level by level in the result
    assert g.active_sets == o.active_sets
    assert (g.n_feasible_lps, g.n_final_lps) == (o.n_feasible_lps, o.n_final_lps)
    r = o.records
    assert st["candidates"] == len(r) and st["opt_lps"] == int((r["feasible"] != 0).sum())
    assert st["pivots_feas"] == int(r["feas_iters"].sum())
    assert st["pivots_p1"] == int(r["p1_iters"].sum()) and st["pivots_p2"] == int(r["p2_iters"].sum())
