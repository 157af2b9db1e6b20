"""Steps of 97 packed rows and more whose projections have an odd number of groups of K, against
the oracle: one group, three, seven and nine (which are split over K), row counts around the
kernel's tiles of 128 rows, MLP widths of an odd and an even number of groups."""
import numpy as np
import pytest

from tests import workloads
from tests.test_gpu_decode_step import _rel_l2, _run_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [97, 128, 129, 257])
@pytest.mark.parametrize("hidden,hq,hkv,d,inter", [
    (128, 1, 1, 128, 128),
    (384, 6, 2, 64, 1024),
    (896, 14, 2, 64, 4864),
    (1152, 9, 3, 128, 1152),
])
def test_rows_and_widths(rows, hidden, hq, hkv, d, inter):
    rng = np.random.default_rng(rows + hidden)
    new = [1, rows - 4, 1, 2]
    cfg, layers, batch = workloads.decode_step_problem(
        rng, num_layers=1, hidden=hidden, hq=hq, hkv=hkv, d=d, inter=inter,
        ctx=[70, rows + 20, 1, 9], new_tokens=new, qkv_bias=bool(rows & 1))
    r, got, want, lay, bat = _run_both(cfg, layers, batch)
    # one layer: the bounds of the 200-row mixed batch (tests/test_gpu_decode_step.py)
    assert _rel_l2(got, want) < 4e-3
    assert np.all(np.abs(got - want) <= 1.2e-2 + 1.6e-2 * np.abs(want))
    assert _rel_l2(r.h.to_numpy(np.float32, bat["h"].shape), bat["h"]) < 4e-3
