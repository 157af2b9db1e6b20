"""Values of keys that a token does not see do not reach it, also where they are not finite: prompt chunks
at 64-wide heads, V rows of some new tokens holding infinities and NaNs.  Every earlier token's row has
the bits of a run without them, every later one's the same in the elements that are finite and no finite
value in the others; the other KV heads are untouched."""
import numpy as np
import pytest

from tests import workloads
from tests.gpu_harness import PagedAttnRunner

pytestmark = pytest.mark.gpu

BAD = {3: np.inf, 17: -np.inf, 40: np.nan, 63: np.inf}  # element of the head -> value


# column groups by key phases, tokens of a wave (32 / group), tiles of 64 keys that tokens end in
@pytest.mark.parametrize("new,prior,hq,hkv", [
    ([40], [30], 14, 2), ([40, 1, 70], [100, 9, 60], 2, 2),     # few columns
    ([200, 3, 331], [15, 90, 0], 14, 2), ([150], [64], 32, 2),  # more
    ([700, 600], [3, 40], 14, 2), ([300], [0], 128, 8),         # many
])
@pytest.mark.parametrize("causal", [True, False])
def test_values_of_unseen_keys(new, prior, hq, hkv, causal):
    rng = np.random.default_rng(sum(new) + hq)
    c = workloads.paged_case(rng, new, prior, hq=hq, hkv=hkv, d=64)
    clean = PagedAttnRunner(c, causal=causal)
    clean.launch()
    want = clean.result().reshape(-1, hq, 64)
    row0, bad_at = 0, []
    for s, (n, p) in enumerate(zip(new, prior)):
        bad = sorted({n - 1, n // 2, n // 3 + 1 if n > 3 else n - 1})
        for i in bad:
            slot = c["block_tables"][s][(p + i) // 16] * 16 + (p + i) % 16
            for e, x in BAD.items():
                c["v_pool"].reshape(-1, hkv, 64)[slot, 0, e] = x
        bad_at += [(row0 + i, bad[0] <= i or not causal) for i in range(n)]
        row0 += n
    r = PagedAttnRunner(c, causal=causal)
    r.launch()
    got = r.result().reshape(-1, hq, 64)
    sees = np.array([b for _, b in bad_at])
    mine, finite = np.arange(hq) < hq // hkv, ~np.isin(np.arange(64), list(BAD))
    assert np.array_equal(got[:, ~mine].view(np.uint16), want[:, ~mine].view(np.uint16))
    assert np.array_equal(got[~sees].view(np.uint16), want[~sees].view(np.uint16))
    assert np.array_equal(got[:, mine][:, :, finite].view(np.uint16), want[:, mine][:, :, finite].view(np.uint16))
    assert not np.isfinite(got[sees][:, mine][:, :, ~finite].astype(np.float32)).any()
