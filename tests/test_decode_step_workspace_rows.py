"""The step's workspace for more rows is never smaller: a caller that sizes it once for its largest batch
has enough for every smaller one."""
import pytest

from logismos_amd import kernels

GEOMETRIES = [  # hidden, query heads, KV heads, head width, MLP width, vocabulary
    (896, 14, 2, 64, 4864, 0), (1536, 12, 2, 128, 8960, 0), (4096, 32, 8, 128, 12288, 151936),
    (384, 3, 1, 128, 640, 0), (2048, 16, 4, 128, 2048, 32000)]


@pytest.mark.parametrize("turbo3", [0, 1])
@pytest.mark.parametrize("seqs", ["every row", 1, 7])
@pytest.mark.parametrize("hidden,hq,hkv,d,inter,vocab", GEOMETRIES)
def test_more_rows_never_need_less(hidden, hq, hkv, d, inter, vocab, seqs, turbo3):
    if turbo3 and d != 128:
        pytest.skip("3-bit head rows are 128 wide")
    cfg = kernels.DecodeConfig(36, hidden, hq, hkv, d, inter, 1e-6, 16, 512, 8192, vocab, turbo3)
    last = 0
    for rows in [*range(1, 300), *range(300, 9000, 97)]:
        need = kernels.decode_step_workspace_bytes_tokens(cfg, rows if seqs == "every row" else min(seqs, rows),
                                                          rows, 8)
        if need == 0 and last:  # (a width the vocabulary projection does not take at these rows)
            assert False, rows
        assert need >= last, rows
        last = need
