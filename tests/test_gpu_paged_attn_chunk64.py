"""Prompt chunks at 64-wide heads (the kernel whose waves take 32 (token, head) columns) against the CPU
oracle, tolerance of the other head widths (2e-3 max-abs or 1e-2 relative): each split of a workgroup's
waves into column groups and key phases, columns around a wave and a workgroup, contexts around a tile
of 64 keys, blocks of 16, 32, 48 and 80 rows, groups of 1 to 16 heads, without the causal mask, tokens
that see no key; and against 64 bits no further off than the rounding of the output and of the
probabilities' two fp16 terms allow."""
import numpy as np
import pytest

from tests import workloads
from tests.gpu_harness import PagedAttnRunner
from tests.test_gpu_paged_attn_head_dims import _check

pytestmark = pytest.mark.gpu


# rows x hq / 128 groups of columns: under a quarter of the compute units, under all of them, more
@pytest.mark.parametrize("new,prior,hq,hkv", [
    ([2, 1, 5, 3], [0, 30, 61, 126], 14, 2),                  # few
    ([33, 1, 18, 64], [31, 4, 110, 1000], 14, 2),
    ([300, 2, 1, 331], [15, 700, 90, 0], 14, 2),              # some
    ([150, 149], [1, 64], 32, 2),
    ([1100, 1, 900, 600], [3, 500, 128, 40], 14, 2),          # many
    ([257, 640], [200, 0], 64, 4),
])
def test_column_groups_and_key_phases(new, prior, hq, hkv):
    rng = np.random.default_rng(sum(new) + hq)
    c = workloads.paged_case(rng, new, prior, hq=hq, hkv=hkv, d=64)
    _check(c, what=f"{new} x {hq}/{hkv}")


@pytest.mark.parametrize("hq,hkv", [(1, 1), (2, 2), (3, 1), (16, 1), (21, 3), (24, 8)])
@pytest.mark.parametrize("block_size", [16, 32, 48, 80])
def test_groups_and_blocks(hq, hkv, block_size):
    rng = np.random.default_rng(hq * 100 + block_size)
    c = workloads.paged_case(rng, [7, 1, 40, 2], [57, 9, 150, 0], hq=hq, hkv=hkv, d=64,
                             block_size=block_size)
    _check(c, what=f"{hq}/{hkv}, blocks of {block_size}")


@pytest.mark.parametrize("rows", [[9, 3, 1], [500, 120, 1]])
def test_without_the_causal_mask(rows):
    rng = np.random.default_rng(rows[0])
    c = workloads.paged_case(rng, rows, [70, 0, 5], hq=14, hkv=2, d=64)
    _check(c, causal=False, what="not causal")


def test_tokens_that_see_no_key():
    # contexts shorter than the new tokens: the first tokens see nothing, rows of zeros
    rng = np.random.default_rng(5)
    c = workloads.paged_case(rng, [40, 6, 1], [30, 2, 8], hq=14, hkv=2, d=64)
    c["context_lens"] = np.array([25, 0, 9], c["context_lens"].dtype)
    r = PagedAttnRunner(c)
    r.launch()
    got = r.result().reshape(-1, 14, 64)
    assert not np.any(got[:15]) and not np.any(got[40:46])
    assert np.all(np.isfinite(got.astype(np.float32))) and np.all(np.any(got[15:40] != 0, axis=2))


def test_error_against_64_bits():
    rng = np.random.default_rng(11)
    new, prior, hq, hkv = [90, 35], [400, 30], 14, 2
    c = workloads.paged_case(rng, new, prior, hq=hq, hkv=hkv, d=64)
    r = PagedAttnRunner(c)
    r.launch()
    got = r.result().astype(np.float64).reshape(-1, hq, 64)
    q = np.asarray(c["q"], np.float64).reshape(-1, hq, 64)
    k, v = (np.asarray(c[n], np.float64).reshape(-1, hkv, 64) for n in ("k_pool", "v_pool"))
    row = 0
    for s, (n, p) in enumerate(zip(new, prior)):
        at = np.concatenate([b * 16 + np.arange(16) for b in c["block_tables"][s][:(n + p + 15) // 16]])
        for i in range(n):
            vis = at[:p + i + 1]
            for h in range(hq):
                sc = k[vis, h // 7] @ q[row + i, h] * c["scale"]
                w = np.exp(sc - sc.max())
                w /= w.sum()
                want, size = w @ v[vis, h // 7], w @ np.abs(v[vis, h // 7])
                # fp16 output; fp32 scores (64 terms) move a weight by at most their rounding
                bound = 2.0 ** -11 * np.abs(want) + 2.0 ** -25 + 2.0 ** -16 * size
                assert np.all(np.abs(got[row + i, h] - want) <= bound)
        row += n
