"""The tiled convolution where it can go wrong: sequence boundaries at every place of a tile and of the four tokens it takes
together, empty sequences (more than 64 inside one tile), both tile lengths, a pool whose address allows no paired state
loads, channel counts that leave threads over; and a layer call whose GDN output lies over the convolution's input, which
keeps the state update before it. Against the CpuOps oracle (outputs within one rounding, states bit for bit)."""
import numpy as np
import pytest

import cases
import oracle
import roost_amd
from test_attention_gpu import from_dev, to_dev
from test_gdn_decode_layer_gpu import Layer
from test_gdn_layer_gpu import BF16_ULP, _conv_case

pytestmark = pytest.mark.gpu

# One rounding of each output (bf16; 2e-5 in f32, exp and reciprocal included), and what fp32 sums leave where the terms cancel (a few of millions of outputs): width + 1
# roundings of partial sums of at most sum |w x| + |bias| (below 16 at these distributions), times SiLU's slope (at most 1.1).
CANCEL = 1.1 * 5 * 2.0 ** -24 * 16


def assert_close(got, want, bf16):
    got, want = (oracle.bf16_to_f64(a) if bf16 else np.asarray(a, np.float64) for a in (got, want))
    bad = ~(np.abs(got - want) <= (BF16_ULP if bf16 else 2e-5) * np.abs(want) + CANCEL)
    assert not bad.any(), f"{bad.sum()} outputs off, e.g. got {got[bad][:4]} want {want[bad][:4]}"

STARTS = [1, 2, 3, 4, 5, 6, 7, 8, 9, 40, 0, 0, 33, 1, 1, 1, 2, 3, 1, 300]       # every offset of a tile, few tokens
EMPTIES = [40] + [0] * 150 + [100] + [0] * 70 + [2, 1, 1] + [0] * 5 + [6000]      # more than 64 ends in one tile
LONG = [5, 400, 1, 0, 2, 1001, 3, 130, 1]                                         # tiles of 8


@pytest.mark.parametrize("lens", [STARTS, EMPTIES, LONG], ids=["starts", "empties", "long"])
@pytest.mark.parametrize("channels,width,bf16,state_f32", [(1032, 4, True, False), (72, 3, True, True),
                                                           (40, 2, True, False), (26, 4, False, True),
                                                           (2052, 4, True, False)])
def test_conv_tile_boundaries(session, lens, channels, width, bf16, state_f32):
    slots = [(7 * i) % (len(lens) + 3) if i % 5 else -1 for i in range(len(lens))]
    slots = [s if slots.index(s) == i or s < 0 else -1 for i, s in enumerate(slots)]
    got, want, got_state, want_state = _conv_case(session, lens, slots, len(lens) + 3, channels, width, True, True, bf16,
                                                  state_f32, channels + width)
    assert_close(got, want, bf16)
    assert np.array_equal(got_state.view(np.uint8), want_state.view(np.uint8)), "conv state not bit-exact"


def test_conv_tile_odd_state_address(session):
    rng = np.random.default_rng(8)
    lens, ch, width = [9, 1, 2, 1, 70, 30], 64, 4
    T, B = sum(lens), len(lens)
    x, w = (cases.bf16_bits(rng.standard_normal(n).astype(np.float32)) for n in (T * ch, ch * width))
    state = cases.bf16_bits(rng.standard_normal(B * ch * 3).astype(np.float32))
    slots, cu = np.arange(B, dtype=np.int32)[::-1].copy(), np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    want, want_state = np.zeros(T * ch, np.uint16), state.copy()
    oracle.causal_conv1d(x, w, None, want, want_state, slots, cu, batch=B, tokens=T, channels=ch, width=width, silu=True)
    pool = to_dev(np.concatenate([np.zeros(1, np.uint16), state]), True)[1:]  # 2 bytes past a 16-byte boundary
    out = to_dev(np.zeros(T * ch, np.uint16), True)
    roost_amd.causal_conv1d(session, to_dev(x, True), to_dev(w, True), None, out, pool, to_dev(slots), to_dev(cu), batch=B,
                            tokens=T, channels=ch, width=width, silu=True)
    assert_close(from_dev(out, True), want, True)
    assert np.array_equal(from_dev(pool, True), want_state)


@pytest.mark.parametrize("whole", [0, 1], ids=["no slot", "one slot"])
@pytest.mark.parametrize("bf16_state", [True, False])
@pytest.mark.parametrize("lens", [[5, 70, 0, 33, 1, 2, 40, 300], [1, 2, 1, 5, 1]], ids=["tiles", "short"])
def test_conv_slots_outside_the_pool(session, lens, bf16_state, whole):
    """A call without history: slots of -1 and beyond a pool that may hold no slot at all (the span ends with it). Absent
    slots read nothing, so the results are those of a zero history and the pool, NaN throughout, stays as it is."""
    rng = np.random.default_rng(len(lens) + whole)
    ch, width, T, B = 2048, 4, sum(lens), len(lens)
    x, w = (cases.bf16_bits(rng.standard_normal(n).astype(np.float32)) for n in (T * ch, ch * width))
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    want, zeros = np.zeros(T * ch, np.uint16), np.zeros(B * ch * 3, np.float32)
    oracle.causal_conv1d(x, w, None, want, zeros, np.arange(B, dtype=np.int32), cu, batch=B, tokens=T, channels=ch,
                         width=width, silu=True)
    slots = np.array([-1 if i % 2 else whole + i for i in range(B)], np.int32)
    nan = np.full(ch * 3, np.nan, np.float32)
    pool = to_dev(cases.bf16_bits(nan), True) if bf16_state else to_dev(nan, False)
    before = pool.clone()
    out = to_dev(np.zeros(T * ch, np.uint16), True)
    p = roost_amd.causal_conv1d_params(to_dev(x, True), to_dev(w, True), None, out, pool, to_dev(slots), to_dev(cu),
                                       batch=B, tokens=T, channels=ch, width=width, silu=True)
    p.conv_state.length = whole * ch * 3
    session.launch(session.lib.entry(roost_amd.CAUSAL_CONV1D_VARIANT), p)
    assert_close(from_dev(out, True), want, True)
    assert from_dev(pool, bf16_state).tobytes() == from_dev(before, bf16_state).tobytes()


def test_layer_output_over_the_convolution_input(session):
    """The GDN output in the convolution's input buffer (dead once the convolution has run): the state update, which reads
    that input, may then not wait for the layer's last launch."""
    rng = np.random.default_rng(21)
    layer = Layer(rng, [70, 1, 17], 2, 2, 4, True, "bf16", True, [0, 2, 1], [1, 0, 2])
    want_out, want_cs, want_st = layer.four_ops(session)
    t = layer.t
    y, _, dout, dcs, dst = layer.buffers()
    conv = layer.conv_params(y, dcs)
    x = conv._keep[0]  # the call's input tensor, whose first rows the GDN output takes
    keep = x.clone()
    o = x.reshape(-1)[:layer.T * layer.vh * 128].reshape(layer.T, layer.vh, 128)
    roost_amd.gdn_layer(session, conv, layer.gates_params(None, None), layer.gdn_params(y, o, dst, None, None),
                        layer.norm_params(o, dout), key="over")
    t.cuda.synchronize()
    out, cs, st = from_dev(dout, True), from_dev(dcs, True), from_dev(dst)
    x.copy_(keep)
    n = layer.T * layer.vh
    assert np.array_equal(out[:n], want_out[:n])
    assert np.array_equal(cs, want_cs)
    assert np.array_equal(st, want_st)
