"""What the decode attention into the prepared layout refuses before it touches the device: head widths
other than 128, also where a step writes that layout itself (heads of 32 and 64), and more than 32
sequences."""
import ctypes as C

import pytest

from logismos_amd import kernels

INVALID_VALUE = 1


def _launch(num_seqs, hq, hkv, d, max_blocks, splits):
    p = C.c_void_p(4096)  # never read: the call is refused
    return kernels.library().logismos_launch_paged_attn_decode_fp16_xprep(
        p, p, p, p, p, p, p, p, num_seqs, hq, hkv, d, 16, max_blocks, splits, 0.125, None)


@pytest.mark.parametrize("d", [32, 64, 96, 256])
@pytest.mark.parametrize("max_blocks,splits", [(16, 1), (16, 4), (200, 8)])
def test_other_head_widths(d, max_blocks, splits):
    assert _launch(2, 8, 2, d, max_blocks, splits) == INVALID_VALUE


def test_more_than_32_sequences():
    assert _launch(33, 8, 2, 128, 200, 8) == INVALID_VALUE
