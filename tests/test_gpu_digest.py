"""The result digest at the edges of its pairs and tiles, against the rows."""
import numpy as np
import pytest

import mnmgdatalog_amd as dlg
from grid_closure import rows_digest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 511, 512, 513, 4095, 4096, 4097, 8191, 8193, 2_100_001])
def test_sizes(n):
    rng = np.random.default_rng(n)
    rows = np.stack([rng.permutation(n) - n // 2, np.full(n, 2**31 - 1)], 1).astype(np.int32)   # its own closure
    with dlg.Ctx(0) as c:
        got = c.run("tc", rows, strategy=1, check_output=1)
    assert got["output_size"] == n and got["output_order_breaks"] == 0
    assert got["output_sum"] == rows_digest(got["rows"])
