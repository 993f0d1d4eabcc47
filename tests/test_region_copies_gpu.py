"""mpqp_regions() outputs through the staging blocks: the same sets repeated
until the outputs fill less than one block, end at a block's edge, need the
copying threads, use every block more than once, or have inputs larger than a
block, come back as the first ones did, each in its array."""
import numpy as np
import pytest

from mpqpcudasolver_amd import load_library, synthetic_mpqp
from mpqpcudasolver_amd.host import REGION_FOUND

pytestmark = pytest.mark.gpu

FIELDS = ("status", "n_rows", "radius", "iters", "center", "parameter_A", "parameter_b", "lagrange_A", "lagrange_b",
          "cr_A", "cr_b")
BLOCK = 4 << 20


def _bytes_per_set(n, m0, p, width):
    return 8 * (n * p + n + width * p + width + m0 * p + m0 + p) + 32


@pytest.mark.parametrize("total", [0, 1, BLOCK - 1, BLOCK, 2 * BLOCK - 1, 2 * BLOCK, 11 * BLOCK, 40 * BLOCK + 5])
@pytest.mark.parametrize("outputs", [True, False])
def test_repeated_sets(total, outputs):
    lib = load_library()
    assert lib.warm_up() == 0, lib.last_error()
    n, m, p = 6, 14, 2
    prog = synthetic_mpqp(n, m, p, 3)
    m0 = prog.A.shape[0] + prog.A_t.shape[0]
    count = -(-total // _bytes_per_set(n, m0, p, n))
    print(f"case: regions n={n} m={m} p={p}, {count} sets, outputs {outputs}", flush=True)
    base = np.full((7, n), -1, dtype=np.intc)
    for i, S in enumerate([[], [0], [3], [1, 5], [0, 2, 7], [4], [2, 9, 11]]):
        base[i, :len(S)] = S
    want = lib.regions(prog, base)
    got = lib.regions(prog, np.resize(base, (count, n)), outputs=outputs)
    st = lib.region_stats()
    assert st["sets"] == count and st["found"] == int((got.status == REGION_FOUND).sum())
    for f in FIELDS:
        a = getattr(got, f)
        if a is None:
            assert not outputs
            continue
        w = getattr(want, f)
        assert np.array_equal(a, w[np.arange(count) % 7], equal_nan=w.dtype.kind == "f"), f
