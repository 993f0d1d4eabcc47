"""mpqp_regions() on both sides of the tableau size at which a set gets 256
threads instead of 128, and at the smallest: every output equals the oracle's
within the tolerances of the region tests."""
import os

import numpy as np
import pytest

from conftest import ROOT
from mpqpcudasolver_amd import load_library, synthetic_mpqp
from oracle_lib import OracleLib
from test_regions_gpu import compare

pytestmark = pytest.mark.gpu


# (n, m, p): (m + 2 p + 1) x (2 p + 3) entries: 20, 1,995, 2,014
@pytest.mark.parametrize("n,m,p", [(1, 1, 1), (12, 88, 8), (12, 89, 8)])
def test_both_thread_counts(n, m, p):
    lib, orc = load_library(), OracleLib(os.path.join(ROOT, "oracle", "_build", "libmpqp_oracle.so"))
    assert lib.warm_up() == 0, lib.last_error()
    print(f"case: regions n={n} m={m} p={p}", flush=True)
    prog = synthetic_mpqp(n, m, p, 3)
    rng = np.random.default_rng(4)
    sets = [[]] + [sorted(rng.choice(m, size=int(rng.integers(1, min(n, 4) + 1)), replace=False).tolist())
                   for _ in range(200)]
    compare(lib.regions(prog, sets), orc.regions(prog, sets), sets)
