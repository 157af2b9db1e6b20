"""What the step executor refuses before anything is launched: a missing or misaligned operand of
any layer, at one row, at sixteen (fused projections) and at seventeen (32-row projections).  The
addresses are made up; only the returned status is looked at."""
import ctypes as C

import pytest

from logismos_amd import kernels

INVALID = 1  # hipErrorInvalidValue
LAYERS = 2


def _step(rows, turbo3):
    cfg = kernels.DecodeConfig(LAYERS, 512, 4, 2, 128, 1024, 1e-6, 16, 8, 128, 0, int(turbo3))
    assert kernels.decode_step_workspace_bytes(cfg, rows, 1) > 0  # the geometry is one it takes
    at = iter(range(1 << 20, 1 << 30, 1 << 16))
    layers = (kernels.DecodeLayer * LAYERS)()
    for L in layers:
        for name in ("qkv", "o", "gate_up", "down"):
            setattr(L, name, kernels.Q4Weight(next(at), next(at), next(at)))
        for name in ("norm1_w_f32", "norm2_w_f32", "k_pool_f16", "v_pool_f16"):
            setattr(L, name, next(at))
    batch = kernels.DecodeBatch(*(next(at) for _ in range(10)), rows, 1)
    return cfg, layers, batch, next(at)


def _status(cfg, layers, batch, workspace):
    return kernels.library().logismos_launch_decode_step(C.byref(cfg), layers, C.byref(batch),
                                                         C.c_void_p(workspace), None)


@pytest.mark.parametrize("turbo3", [False, True])
@pytest.mark.parametrize("rows", [1, 16, 17])
def test_missing_operand(rows, turbo3):
    fields = [("batch", n) for n in ("hidden_f32", "final_norm_w_f32", "block_tables", "cu_seqlens",
                                     "context_lens", "positions", "slot_mapping", "rope_cos_f32",
                                     "rope_sin_f32")]
    fields += [(i, n) for i in range(LAYERS)
               for n in ("norm1_w_f32", "norm2_w_f32", "k_pool_f16", "v_pool_f16")]
    for where, name in fields:
        cfg, layers, batch, ws = _step(rows, turbo3)
        setattr(batch if where == "batch" else layers[where], name, None)
        assert _status(cfg, layers, batch, ws) == INVALID, (where, name)


@pytest.mark.parametrize("rows", [1, 16, 17])
@pytest.mark.parametrize("projection", ["qkv", "o", "gate_up", "down"])
def test_missing_or_misaligned_weight(rows, projection):
    for layer in range(LAYERS):
        for part in ("qw", "scale", "zero"):
            cfg, layers, batch, ws = _step(rows, False)
            setattr(getattr(layers[layer], projection), part, None)
            assert _status(cfg, layers, batch, ws) == INVALID, (layer, part)
        for off in (1, 4, 8):
            cfg, layers, batch, ws = _step(rows, False)
            getattr(layers[layer], projection).qw += off
            assert _status(cfg, layers, batch, ws) == INVALID, (layer, off)
