"""A step of one row, whose layers are one resident launch (decode_resident.hip): edges of its lists and
pieces against the oracle, any number of workgroups bit for bit, and against the route of 2 to 16 rows."""
import copy
import ctypes as C

import numpy as np
import pytest

import oracle as O
from logismos_amd import hip, kernels
from oracle import decode_step as OS
from tests import workloads
from tests.gpu_harness import DecodeStepRunner, PagedAttnRunner
from tests.test_gpu_decode_step import _rel_l2

pytestmark = pytest.mark.gpu

SHAPES = [  # hidden, query heads, KV heads, head width, MLP width, context, rows per KV block
    (128, 1, 1, 128, 128, 1, 16),          # one group of K: seven waves with nothing; parts without a tile
    (384, 3, 3, 128, 256, 16, 32),         # a whole tile of keys
    (896, 14, 2, 64, 4864, 17, 16),        # 7 and 38 groups: shares of four and one; the new key alone in its tile
    (896, 14, 2, 64, 4864, 500, 48),       # four pieces, read by the o projection itself
    (1536, 12, 2, 128, 8960, 129, 16),     # 12 and 70 groups: shares of two and one, nine; one piece and a key
    (512, 16, 1, 64, 512, 1300, 16),       # the widest group of heads, eleven pieces merged
    (2176, 17, 17, 128, 1152, 700, 16),    # no two heads share K and V; more than one tile per wave
    (4096, 32, 8, 128, 1024, 2100, 16),    # the widest norm, seventeen pieces merged
    (512, 8, 2, 64, 16384, 70, 64),        # the widest operand
    (512, 64, 8, 128, 512, 100, 16),       # one piece of a group's eight heads: 56 workgroups that merge a head have
                                           # q/k/v tiles and no piece of the context
    (512, 8, 2, 64, 512, 1000, 16),        # eight pieces, read by the o projection itself in two rounds
    (512, 24, 8, 64, 512, 500, 16),        # the most columns of heads that are read so
]


def _problem(shape, layers=1, seed=0, bias=True):
    hidden, hq, hkv, d, inter, ctx, block = shape
    return workloads.decode_step_problem(
        np.random.default_rng(seed + hidden + ctx), num_layers=layers, hidden=hidden, hq=hq, hkv=hkv, d=d,
        inter=inter, ctx=[ctx], block_size=block, qkv_bias=bias)


def _state(r, batch, layers):
    out = r.result_bits().copy()
    h = r.h.to_numpy(np.float32, batch["h"].shape)
    pools = [[b.to_numpy(np.uint16, L["k_pool"].shape) for b in kv] for kv, L in zip(r.pools, layers)]
    return out, h, pools


def _lib():
    # library-internal: size of the region, and the launch with limits of its own
    lib = C.CDLL(kernels.library()._name)
    size = lib.lg_decode_resident_bytes
    size.restype = C.c_size_t

    def launch(cfg, layers, batch, region, workgroups=0, polls=0, tickets=0):
        limits = (C.c_int * 3)(workgroups, polls, tickets)
        return lib.lg_decode_resident_launch(cfg, layers, batch, region, limits, None)
    return size, launch


class OneLaunch(DecodeStepRunner):
    """A step of one row whose layers are one launch whether that pays or not."""

    def __init__(self, cfg, layers, batch, **kw):
        super().__init__(cfg, layers, batch, **kw)
        self.ws = hip.DeviceBuffer(self.ws.nbytes + _lib()[0](C.byref(self.cfg)))
        self.ws.fill(0xFF)

    def launch(self):
        lib = C.CDLL(kernels.library()._name)
        assert lib.lg_launch_decode_step_one_launch(C.byref(self.cfg), self.layers, C.byref(self.batch), self.ws.ptr,
                                                    self.stream.raw if self.stream else None) == 0


def _run_both(cfg, layers, batch):
    r = OneLaunch(cfg, layers, batch)
    r.launch()
    got = O.bf16_bits_to_f32(r.result_bits())
    lay, bat = copy.deepcopy(layers), dict(batch, h=batch["h"].copy())
    return r, got, O.bf16_bits_to_f32(OS.decode_step(cfg, lay, bat)), lay, bat


@pytest.mark.parametrize("shape", SHAPES)
def test_against_the_oracle(shape):
    cfg, layers, batch = _problem(shape)
    r, got, want, lay, bat = _run_both(cfg, layers, batch)
    # one layer: the decode batch's bounds (tests/test_gpu_decode_step.py)
    assert _rel_l2(got, want) < 6e-3
    assert np.all(np.abs(got - want) <= 1.5e-2 + 2e-2 * np.abs(want))
    assert _rel_l2(r.h.to_numpy(np.float32, bat["h"].shape), bat["h"]) < 6e-3
    for (kp, vp), L in zip(r.pools, lay):
        for buf, ref in ((kp, L["k_pool"]), (vp, L["v_pool"])):
            diff = np.abs(buf.to_numpy(np.float16, ref.shape).astype(np.float32) - ref.astype(np.float32))
            assert np.all((diff <= 4e-3) | (diff <= 1e-2 * np.abs(ref.astype(np.float32))))


@pytest.mark.parametrize("workgroups", [1, 7, 100, 255])
@pytest.mark.parametrize("shape", [SHAPES[2], (512, 8, 2, 128, 1024, 900, 16), SHAPES[9]])
def test_any_number_of_workgroups(shape, workgroups):
    # the work is cut for all compute units; fewer workgroups take several parts each, phase by phase
    cfg, layers, batch = _problem(shape, layers=3)
    whole = OneLaunch(cfg, layers, batch)
    size, launch = _lib()
    want = None
    for n in (0, workgroups, workgroups):
        r = DecodeStepRunner(cfg, layers, batch)
        region = hip.DeviceBuffer(size(C.byref(r.cfg)))
        region.fill(0xFF)
        assert launch(C.byref(r.cfg), r.layers, C.byref(r.batch), region.ptr, n) == 0
        hip.synchronize()
        got = _state(r, batch, layers)
        want = want or got
        assert np.array_equal(got[1], want[1])
        assert all(np.array_equal(a, b) for x, y in zip(got[2], want[2]) for a, b in zip(x, y))
    whole.launch()
    assert np.array_equal(_state(whole, batch, layers)[1], want[1])


@pytest.mark.parametrize("shape", [SHAPES[2], (512, 8, 2, 128, 1024, 900, 16), SHAPES[9]])
def test_closed_before_all_workgroups_are_there(shape):
    # the step is closed to the first so many that hold tickets, as after a wait for the others: those leave
    cfg, layers, batch = _problem(shape, layers=3)
    size, launch = _lib()
    table = (3 * 136 + 255) // 256 * 256  # in front of the region: three layers' operands
    want = None
    for tickets in (0, 255, 100, 7, 1):
        r = DecodeStepRunner(cfg, layers, batch)
        region = hip.DeviceBuffer(size(C.byref(r.cfg)))
        region.fill(0xFF)
        assert launch(C.byref(r.cfg), r.layers, C.byref(r.batch), region.ptr, tickets=tickets) == 0
        hip.synchronize()
        assert region.to_numpy(np.uint32, (3,), table).tolist() == [256, tickets or 256, 0]
        got = _state(r, batch, layers)
        want = want or got
        assert np.array_equal(got[1], want[1])
        assert all(np.array_equal(a, b) for x, y in zip(got[2], want[2]) for a, b in zip(x, y))


def test_beside_another_stream():
    # prompt attention on another stream holds compute units for longer than a step waits for them
    cfg, layers, batch = _problem(SHAPES[2], layers=3)
    alone = OneLaunch(cfg, layers, batch)
    alone.launch()
    want = _state(alone, batch, layers)
    other = PagedAttnRunner(workloads.paged_case(np.random.default_rng(1), [64], [20000], hq=32, hkv=8,
                                                 pool_period_rows=4096), stream=hip.Stream())
    stream = hip.Stream()
    steps = [OneLaunch(cfg, layers, batch, stream=stream) for _ in range(6)]
    hip.synchronize()
    for _ in range(10):
        other.launch()
    for r in steps:
        r.launch()
    hip.synchronize()
    for r in steps:
        got = _state(r, batch, layers)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])


@pytest.mark.parametrize("slot", ["its own", "none", "another key's"])
@pytest.mark.parametrize("shape", [SHAPES[3], (512, 8, 2, 128, 1024, 300, 16)])
def test_against_the_route_of_more_rows(shape, slot):
    # scales off 16 bytes take the fused launches of 2 to 16 rows.  The row may be appended nowhere, or
    # where an earlier key stands: attention then sees what the pools hold.
    cfg, layers, batch = _problem(shape, seed=5)
    if slot != "its own":
        table, bs = batch["block_tables"][0], cfg["block_size"]
        batch["slots"] = np.array([-1 if slot == "none" else int(table[2]) * bs + 5], np.int64)
    states = []
    for off in (0, 4):
        r = (DecodeStepRunner if off else OneLaunch)(cfg, layers, batch)
        if off:
            for lay, L in zip(r.layers, layers):
                s = np.ascontiguousarray(L["qkv"][1]).view(np.uint16).reshape(-1)
                buf = hip.DeviceBuffer.from_numpy(np.concatenate([np.zeros(off // 2, np.uint16), s]))
                r.keep.append(buf)
                w = lay.qkv
                lay.qkv = kernels.Q4Weight(w.qw, buf.ptr.value + off, w.zero)
        r.launch()
        states.append(_state(r, batch, layers))
    (a, ha, pa), (b, hb, pb) = states
    # the same operands and roundings, other orders of the fp32 sums: last bits of fp16 and bf16 values
    assert _rel_l2(ha, hb) < 2e-3
    for x, y, L in zip(pa, pb, layers):
        for u, v, name in zip(x, y, ("k_pool", "v_pool")):
            was = L[name].view(np.uint16)
            changed = np.nonzero((u != was).any(axis=1))[0]
            assert changed.tolist() == ([] if slot == "none" else [int(batch["slots"][0])])
            assert np.allclose(u.view(np.float16).astype(np.float32), v.view(np.float16).astype(np.float32),
                               atol=4e-3, rtol=4e-3)


@pytest.mark.parametrize("hq,hkv,d,mib", [(8, 2, 128, 512), (8, 4, 64, 320), (4, 4, 128, 320)])
def test_tables_too_long_for_one_launch(hq, hkv, d, mib):
    # past so many bytes of K and V that a layer's table can hold a step is launched operator by operator
    cfg, layers, batch = _problem((512, hq, hkv, d, 512, 200, 16), layers=4)
    blocks = (mib << 20) // (4 * hkv * d * 16)
    states = []
    for more in (0, 1):
        b = dict(batch)
        b["block_tables"] = np.full((1, blocks + more), 0x3FFFFFF, np.int32)
        b["block_tables"][0, :13] = batch["block_tables"][0, :13]
        for name in ("cos", "sin"):
            b[name] = np.resize(batch[name], (b["block_tables"].shape[1] * 16, d // 2))
        r = DecodeStepRunner(cfg, layers, b)
        assert C.CDLL(kernels.library()._name).lg_decode_resident_pays(C.byref(r.cfg)) == (more == 0)
        for call in (kernels.launch_decode_step, kernels.launch_decode_step_per_operator):
            r.h.copy_from_host(batch["h"].astype(np.float32))
            call(r.cfg, r.layers, r.batch, r.ws)
            states.append(_state(r, b, layers))
    assert _rel_l2(states[0][1], states[1][1]) < 2e-3
    assert np.array_equal(states[2][1], states[3][1]) and np.array_equal(states[2][0], states[3][0])


@pytest.mark.parametrize("hidden,layers,pays", [(512, 3, 0), (512, 4, 1), (512, 49, 1), (1536, 4, 1), (1664, 15, 0), (1664, 16, 1)])
def test_few_layers_are_launched_operator_by_operator(hidden, layers, pays):
    cfg, lay, batch = _problem((hidden, 4, 2, 64, 256, 40, 16), layers=layers)
    r = DecodeStepRunner(cfg, lay, batch)
    assert C.CDLL(kernels.library()._name).lg_decode_resident_pays(C.byref(r.cfg)) == pays
    states = []
    for call in (r.launch, lambda: kernels.launch_decode_step_per_operator(r.cfg, r.layers, r.batch, r.ws),
                 OneLaunch.launch):
        if call == OneLaunch.launch:
            r = OneLaunch(cfg, lay, batch)
            call = r.launch
        r.h.copy_from_host(batch["h"].astype(np.float32))
        call()
        states.append(_state(r, batch, lay)[1])
    # the route that it takes bit for bit (24 layers' operands are handed over by a launch); the other is last bits of
    # bf16 values away, through the layers
    assert np.array_equal(states[0], states[2 if pays else 1])
    assert _rel_l2(states[1], states[2]) < 1e-2


@pytest.mark.parametrize("rows", [1, 2, 16, 40])
def test_a_launch_per_operator(rows):
    # at one row the route of 2 to 16 rows (what scales off 16 bytes take, bit for bit), otherwise the same step
    cfg, layers, batch = workloads.decode_step_problem(
        np.random.default_rng(rows), num_layers=4, hidden=512, hq=8, hkv=2, inter=768, ctx=[300] * rows, qkv_bias=True)
    states = []
    for per_operator in (False, True):
        r = DecodeStepRunner(cfg, layers, batch)
        if rows == 1 and not per_operator:
            for lay, L in zip(r.layers, layers):
                s = np.ascontiguousarray(L["o"][1]).view(np.uint16).reshape(-1)
                buf = hip.DeviceBuffer.from_numpy(np.concatenate([np.zeros(2, np.uint16), s]))
                r.keep.append(buf)
                lay.o = kernels.Q4Weight(lay.o.qw, buf.ptr.value + 4, lay.o.zero)
        call = kernels.launch_decode_step_per_operator if per_operator else kernels.launch_decode_step
        call(r.cfg, r.layers, r.batch, r.ws)
        out = r.result_bits().copy()
        states.append((out, r.h.to_numpy(np.float32, batch["h"].shape), r.pools))
    (a, ha, pa), (b, hb, pb) = states
    assert np.array_equal(a, b) and np.array_equal(ha, hb)
    for x, y, L in zip(pa, pb, layers):
        for u, v in zip(x, y):
            assert np.array_equal(u.to_numpy(np.uint16, L["k_pool"].shape), v.to_numpy(np.uint16, L["k_pool"].shape))


def test_no_key_is_seen():
    # a context of 0: attention adds nothing, and the layers still follow one another (more workgroups have
    # q/k/v tiles than tiles of the other projections); twice the same, and what a launch per operator gives
    cfg, layers, batch = _problem((1024, 32, 16, 128, 128, 9, 16), layers=4, seed=9)
    batch["context_lens"] = np.zeros(1, np.int32)
    states = []
    for _ in range(2):
        r = OneLaunch(cfg, layers, batch)
        r.launch()
        states.append(_state(r, batch, layers))
    r = DecodeStepRunner(cfg, layers, batch)
    kernels.launch_decode_step_per_operator(r.cfg, r.layers, r.batch, r.ws)
    (a, ha, pa), (b, hb, pb), (_, want, pw) = states[0], states[1], _state(r, batch, layers)
    assert np.array_equal(ha, hb) and np.array_equal(a, b)
    # without attention only the MLPs add to the residual stream: one layer's bound, of four independently
    assert _rel_l2(ha, want) < 4e-3 and _rel_l2(want, batch["h"]) > 0.05
    for x, y in zip(pa, pw):
        for u, v in zip(x, y):
            assert np.allclose(u.view(np.float16).astype(np.float32), v.view(np.float16).astype(np.float32),
                               atol=8e-3, rtol=8e-3)


@pytest.mark.parametrize("shape", [(384, 3, 3, 128, 256, 80, 16), (512, 16, 1, 64, 512, 1296, 16)])
def test_a_context_past_the_block_table(shape):
    # context_lens is a device value that the host does not see: the lists of K/V tiles, whose room follows from
    # the block table, take the keys that the table holds
    states = []
    for past in (0, 1, 100, 10 ** 6):
        cfg, layers, batch = _problem(shape, layers=2)
        assert batch["block_tables"].shape[1] * cfg["block_size"] == shape[5]
        batch["context_lens"] = batch["context_lens"] + np.int32(past)
        r = DecodeStepRunner(cfg, layers, batch)
        size = _lib()[0](C.byref(r.cfg))
        region = hip.DeviceBuffer(size + 4096)
        region.fill(0x5A)
        assert _lib()[1](C.byref(r.cfg), r.layers, C.byref(r.batch), region.ptr) == 0
        hip.synchronize()
        assert (region.to_numpy(np.uint8, (4096,), size) == 0x5A).all()
        states.append(_state(r, batch, layers))
    for got in states[1:]:
        assert np.array_equal(got[1], states[0][1])
        assert all(np.array_equal(a, b) for x, y in zip(got[2], states[0][2]) for a, b in zip(x, y))


@pytest.mark.parametrize("shape", [SHAPES[3], SHAPES[5], SHAPES[7], SHAPES[9]])
def test_a_wait_that_runs_out_shows(shape):
    # every wave gives up at its first poll that does not find its words
    cfg, layers, batch = _problem(shape, layers=3, bias=False)
    r = DecodeStepRunner(cfg, layers, batch)
    size, launch = _lib()
    region = hip.DeviceBuffer(size(C.byref(r.cfg)))
    assert launch(C.byref(r.cfg), r.layers, C.byref(r.batch), region.ptr, polls=1) == 0
    hip.synchronize()
    _, h, pools = _state(r, batch, layers)
    assert np.isnan(h).all()
    slot = int(batch["slots"][0])
    for kv, L in zip(pools, layers):
        for got, name in zip(kv, ("k_pool", "v_pool")):
            assert not np.isnan(got.view(np.float16)).any()
            assert set(np.nonzero((got != L[name].view(np.uint16)).any(axis=1))[0]) <= {slot}
    # the next step over the same region is a step like any other
    want = OneLaunch(cfg, layers, batch)
    want.launch()
    r.h.copy_from_host(batch["h"].astype(np.float32))
    assert launch(C.byref(r.cfg), r.layers, C.byref(r.batch), region.ptr) == 0
    hip.synchronize()
    assert np.array_equal(_state(r, batch, layers)[1], _state(want, batch, layers)[1])


@pytest.mark.parametrize("shape", [SHAPES[3], (512, 8, 2, 128, 512, 1300, 16), (512, 16, 1, 64, 512, 1300, 16)])
def test_pieces_of_keys_that_have_no_weight(shape):
    # every key of the first piece, then of all but the last two, has a score of -inf (K minus infinity where the
    # queries are far above zero): such a piece weighs nothing beside the others, in whatever order they meet
    hidden, hq, hkv, d, inter, ctx, block = shape
    for keys in (128, ctx - 2):
        cfg, layers, batch = _problem(shape, seed=11)
        batch["cos"], batch["sin"] = np.ones_like(batch["cos"]), np.zeros_like(batch["sin"])
        L = layers[0]
        L["qkv_bias"][:hq * d:d] = 100.0
        key = np.arange(keys)
        rows = batch["block_tables"][0][key // block].astype(np.int64) * block + key % block
        L["k_pool"][rows[:, None], np.arange(hkv) * d] = -np.inf
        r, got, want, _, bat = _run_both(cfg, layers, batch)
        assert np.isfinite(want).all() and np.isfinite(got).all()
        assert _rel_l2(got, want) < 6e-3
        assert _rel_l2(r.h.to_numpy(np.float32, bat["h"].shape), bat["h"]) < 6e-3
