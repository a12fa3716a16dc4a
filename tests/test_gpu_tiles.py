"""The tiles of the expert projections at the sizes where they can go wrong, against the CPU oracle:
experts that end at and around the edges of a tile's rows, K shorter than the ring of stages, output
widths that are no multiple of a tile, the smallest and largest row counts of a variant's range."""
import numpy as np
import pytest
import torch
from scipy.special import erfc

import aristos_amd as ka
from aristos_amd import synth
from helpers import pack_inputs, random_layer
from oracle import moe_ref
from test_gpu_parity import MODE_IDS, MODES, _apply, _keys, _one_hot_layer, _out_to_np, _to_device, check_against_oracle, run_gpu

pytestmark = pytest.mark.gpu


def _forced_rows(dt, H, I, rows, cf, mode, act=1):
    """One launch of a layer whose expert e is routed rows[e] tokens (k = 1)."""
    S = -(-sum(rows) // 128) * 128
    rows = list(rows) + [S - sum(rows)] if S > sum(rows) else list(rows)
    keys = _keys(S, H, I, len(rows), 1, cf=cf, act=act, dt=dt)
    c = moe_ref.cfg_from_keys(keys)
    iP = _one_hot_layer(c, rows, seed=31 + H + I)
    d, v, _, _ = check_against_oracle(c, keys, iP, mode)
    np.testing.assert_array_equal(v["expert_count"], np.array(rows))
    return d


@pytest.mark.parametrize("mode", MODES, ids=MODE_IDS)
@pytest.mark.parametrize("dt", [0, 1], ids=["fp32", "tf32"])
@pytest.mark.parametrize("H,I", [(64, 64), (128, 320), (448, 192)])
def test_32_bit_tiles_at_the_edges_of_their_rows(mode, dt, H, I):
    """64-row tiles of two wavefront rows of 32, over two K slices (fewer than the ring holds) and more."""
    _forced_rows(dt, H, I, [1, 31, 32, 33, 63, 64, 65, 95, 97, 127, 128, 129, 160, 5], cf=4.0, mode=mode)


@pytest.mark.parametrize("mode", MODES, ids=MODE_IDS)
@pytest.mark.parametrize("S,H,I,E,act", [(16384, 320, 320, 64, 0), (4096, 1088, 1152, 16, 1)])
def test_tf32_tiles_on_the_bf16_matrix_cores(mode, S, H, I, E, act):
    """256 x 256 tiles, whose operands are scaled to fp16 in LDS: experts that end around the 128 rows of a wavefront
    row and the 256 of a tile, a last column tile of 64 and of 128 columns, K of ten slices and more. The
    products are exact and summed in fp32 as on the fp32 matrix cores: the bounds are those of the other tiles. (The same
    layers with operands that do not fit fp16: test_tf32_tiles_that_are_scaled_anew_or_computed_again.)"""
    edges = [1, 16, 17, 127, 128, 129, 130, 255, 256, 257, 300, 384, 385, 512]
    share, rest = divmod(S - sum(edges), E - len(edges))
    rows = edges + [share + 1] * rest + [share] * (E - len(edges) - rest)
    _forced_rows(1, H, I, rows, cf=2.0, mode=mode, act=act)


@pytest.mark.parametrize("where", ["x", "w_up", "w_down"])
def test_tf32_infinities_on_the_bf16_matrix_cores(where):
    """An infinite operand, which sends its tiles through the bf16 products, against operands whose remainder is zero there (all
    are bf16 values): infinities and NaN in the places where sums of the undivided products have them, and everything else as it is."""
    S, H, I = 16384, 512, 512
    rng = np.random.default_rng(7)
    x, w_up, w_down = (torch.from_numpy(rng.standard_normal(n)).to(torch.bfloat16).float() for n in ((S, H), (I, H), (H, I)))
    w_up, w_down = w_up / 16, w_down / 16
    if where == "x":
        x[300, 17], x[5000, 500], x[16383, 3] = float("inf"), -float("inf"), float("nan")
    elif where == "w_up":
        w_up[200, 33], w_up[500, 511] = float("inf"), -float("inf")
    else:
        w_down[70, 100], w_down[400, 0] = -float("inf"), float("inf")
    iP = torch.cat([x.flatten(), w_up.flatten(), w_down.flatten(), torch.zeros(H + I)]).cuda()
    ka.initialize(_keys(S, H, I, 1, 1, act=0, dt=1))
    try:
        oP = torch.zeros(S * H, device="cuda")
        ka.moe.forward_host_dense(iP, oP)
        ka.moe.stream_synchronize()
        got = oP.view(S, H).cpu().double()
    finally:
        ka.finalize()
    h = x.double() @ w_up.double().T
    h = torch.where(h > 0, h, torch.zeros((), dtype=h.dtype))   # NaN gives 0, as in the kernels
    want = h @ w_down.double().T
    for places in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(places(got), places(want))
    ok = torch.isfinite(want)
    # h is rounded to 11 bits on the way, 2^-11 of each of its values at most, and truncated to as many: nothing on top
    assert float((got - want)[ok].norm()) <= 2.0 ** -11 * float(want[ok].norm()) + 1e-5 * float(want[ok].norm())


@pytest.mark.parametrize("mode", MODES, ids=MODE_IDS)
@pytest.mark.parametrize("dt", [2, 3], ids=["bf16", "fp16"])
@pytest.mark.parametrize("H,I,rows,cf", [
    (64, 64, [1, 15, 16, 17, 31, 32, 33, 47, 63, 64, 65, 40, 30, 40, 20, 30], 2.0),          # 128-row tiles, one K slice: the second group has none
    (192, 320, [1, 15, 16, 17, 31, 32, 33, 47, 63, 64, 65, 40, 30, 40, 20, 30], 2.0),        # three and five slices, a last column tile of 64
    (320, 448, [1, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256, 100, 60, 90, 130], 3.0),   # 64-row tiles, two row blocks and more
    (1152, 1216, [1, 63, 64, 65, 111, 112, 113, 127, 128, 129, 200, 256, 257, 150, 140, 130], 3.0),   # 128-row tiles
    (1152, 64, [128, 120, 130, 126, 129, 127, 128, 128, 64, 100, 255, 1, 128, 128, 160, 162], 3.0),    # 128-row tiles, one K slice down
], ids=["64x64", "192x320", "320x448", "1152x1216", "1152x64"])
def test_tiles_whose_k_is_halved_between_two_groups(mode, dt, H, I, rows, cf):
    """The small tiles of layers with few tiles: each half of K on four wavefronts, the halves added in LDS."""
    _forced_rows(dt, H, I, rows, cf=cf, mode=mode)


@pytest.mark.parametrize("dt", [0, 2, 3], ids=["fp32", "bf16", "fp16"])
def test_gelu_over_the_range_of_its_argument(dt):
    """Both projections the identity, no biases: the layer's output is the activation of its input. In 32 bits it is
    v Phi(v) within |v| 2.5e-7 (the rounding of 1 - Phi(-v), the fit's 1.4e-7) and, below zero, within 1e-5 of itself
    (the rounding of v^2 / 2 <= 50 in the exponent); 16-bit Elements round that once more, on the way in exactly."""
    S, H = 512, 64
    v = np.concatenate([np.linspace(-10.0, 10.0, S * H - 64), np.geomspace(1e-30, 1e4, 32), -np.geomspace(1e-30, 1e4, 32)])
    torch_dt = {0: torch.float32, 2: torch.bfloat16, 3: torch.float16}[dt]
    x = torch.from_numpy(v).to(torch_dt)
    eye = torch.eye(H, dtype=torch_dt)
    iP = torch.cat([x, eye.flatten(), eye.flatten(), torch.zeros(2 * H, dtype=torch_dt)]).cuda()
    ka.initialize(_keys(S, H, H, 1, 1, act=1, dt=dt))
    try:
        oP = torch.full((S * H,), float("nan"), dtype=torch_dt, device="cuda")
        ka.moe.forward_host_dense(iP, oP)
        ka.moe.stream_synchronize()
        got = oP.cpu().double().numpy()
    finally:
        ka.finalize()
    v = x.double().numpy()
    want = v * 0.5 * erfc(-v / np.sqrt(2.0))
    unit, tiny = {0: (0.0, 1e-37), 2: (2.0 ** -8, 1e-37), 3: (2.0 ** -11, 2.0 ** -24)}[dt]   # half a place of 8 and of 11 bits; fp16's last subnormal
    bound = 2.5e-7 * np.abs(v) + 1.001 * unit * np.abs(want) + tiny
    assert (np.abs(got - want) <= bound).all()
    low = (v < 0) & (v > -9.0)
    assert (np.abs(got - want)[low] <= (1e-5 + 1.001 * unit) * np.abs(want[low]) + tiny).all()


@pytest.mark.parametrize("dt,S,H,I,E", [
    (2, 128, 2048, 192, 8),       # eight workgroups a tile, one share each
    (2, 1024, 1984, 192, 64),     # four a tile, shares of 7 and 8 steps; the sums of all 64 experts
    (3, 2048, 2112, 64, 33),      # two a tile, three expert groups of which the last holds one expert
    (0, 128, 512, 64, 8),         # four a tile of four shares
    (1, 512, 576, 64, 24),
    (0, 512, 960, 64, 150),       # 64 experts at a time, the fourth part past the padded count
    (0, 1152, 512, 64, 100),      # two parts, a last round of workgroups
], ids=lambda v: str(v))
def test_gate_tiles_spread_over_workgroups_keep_their_bits(dt, S, H, I, E):
    """Few tokens: the shares of a tile's logits on several workgroups, summed by the last to arrive. Against the phased
    mode, whose workgroups hold all shares, bit for bit, in several launches on the same counters."""
    keys = _keys(S, H, I, E, 2, dt=dt)
    c = moe_ref.cfg_from_keys(keys)
    iP = pack_inputs(c, *random_layer(c, seed=S + E, w_std=0.05, bias_std=0.1))
    _, v0, out0, _ = check_against_oracle(c, keys, iP, ka.MODE_PHASED)
    _, v1, out1, _ = check_against_oracle(c, keys, iP, ka.MODE_FUSED, launches=3)
    for name in ("logits", "topk_expert", "topk_prob", "topk_slot", "expert_count"):
        np.testing.assert_array_equal(v0[name], v1[name])
    np.testing.assert_array_equal(out0, out1)


@pytest.mark.parametrize("dt,S,H,I,E", [
    (2, 2176, 1024, 64, 16),      # 136 tiles, workgroups without one
    (3, 4096, 64, 64, 33),        # a tile for every workgroup; shares of no step and of one
    (2, 4096, 2112, 64, 64),
    (2, 4224, 192, 64, 8),        # one tile more than workgroups have groups of wavefronts for: units of two
], ids=lambda v: str(v))
def test_gate_tiles_one_to_a_workgroup(dt, S, H, I, E):
    """As many tiles as workgroups or a little fewer, against the units of two tiles of the phased mode, bit for bit."""
    test_gate_tiles_spread_over_workgroups_keep_their_bits(dt, S, H, I, E)


@pytest.mark.parametrize("dt,S,H,E,k", [
    (0, 512, 64, 65, 3),          # whole units in both modes; one expert past the first run of 64
    (1, 384, 64, 128, 128),       # every expert picked by every token
    (0, 256, 64, 129, 8),         # a third run of 64 that holds one expert
    (1, 256, 64, 256, 5),
    (0, 256, 512, 127, 4),        # spread over workgroups in the persistent launch
    (1, 128, 1024, 256, 256),
], ids=lambda v: str(v))
def test_gate_of_many_experts_in_32_bits(dt, S, H, E, k):
    """65 to 256 experts of 32-bit Elements: a block of 16 tokens by a group of four wavefronts. Against the oracle, the same bits
    in both modes, and the gate's loss of a training step: sums over S probabilities, rounded in fp32, S 2^-24 = 3e-5 at most."""
    keys = _keys(S, H, 64, E, k, dt=dt)
    keys.is_training = 1
    c = moe_ref.cfg_from_keys(keys)
    iP = pack_inputs(c, *random_layer(c, seed=S + E, w_std=0.05, bias_std=0.1))
    got = []
    for mode in MODES[:2]:
        d, v, out, _ = check_against_oracle(c, keys, iP, mode)
        got.append((v, out))
    for name in ("logits", "topk_expert", "topk_prob", "topk_slot", "expert_count"):
        np.testing.assert_array_equal(got[0][0][name], got[1][0][name])
    np.testing.assert_array_equal(got[0][1], got[1][1])
    ref = moe_ref.gate_loss(c, moe_ref.route(c, got[0][0]["logits"])["probs"], got[0][0]["expert_count"])
    ka.initialize(keys)
    try:
        ka.moe.forward_host(_to_device(c, iP), synth.alloc_outputs(d))
        ka.moe.stream_synchronize()
        g = ka.moe.gate_loss(d.E)
    finally:
        ka.finalize()
    assert abs(g["loss"] - ref["loss"]) <= 3e-5 * ref["loss"]
    np.testing.assert_allclose(g["mean_prob"], ref["mean_prob"], rtol=3e-5, atol=1e-8)


@pytest.mark.parametrize("dt,S,H,E,k", [
    (0, 256, 64, 257, 32),        # a second pass that holds one expert; the most picks
    (1, 4224, 128, 384, 3),       # several units to a workgroup
    (0, 128, 1024, 512, 5),
    (2, 384, 128, 300, 3),        # 16-bit: the sums of the product
    (3, 128, 1152, 512, 32),
], ids=lambda v: str(v))
def test_gate_of_more_than_256_experts(dt, S, H, E, k):
    test_gate_of_many_experts_in_32_bits(dt, S, H, E, k)


@pytest.mark.parametrize("dt,S,E,k", [
    (2, 8320, 65, 2),             # a workgroup's slot tiles by four groups of two wavefronts; queues of eight experts, one of nine
    (2, 4224, 128, 3),            # by two groups of four; every queue full
    (3, 128, 256, 8),             # by the whole workgroup, two threads per expert's counts
    (2, 640, 257, 2),             # more experts than a group of the gate takes
    (2, 1152, 512, 4),            # a thread per expert's counts, queues of 64 experts
    (0, 4224, 96, 2),             # workgroups of four wavefronts, two queues each
    (1, 1152, 300, 5),            # more experts than threads
], ids=lambda v: str(v))
def test_slots_and_queues_of_many_experts(dt, S, E, k):
    """Above 64 experts the counts of a slot tile are shared out over a group's threads and the queues are made a wavefront
    each: slots against the oracle, the same bits in every launch mode and under both schedules."""
    keys = _keys(S, 64, 64, E, k, cf=1.25, dt=dt)
    c = moe_ref.cfg_from_keys(keys)
    iP = pack_inputs(c, *random_layer(c, seed=S + E, w_std=0.05, bias_std=0.1))
    got = [check_against_oracle(c, keys, iP, mode, launches=2)[1:3] for mode in MODES]
    for v, out in got[1:]:
        for name in ("topk_slot", "expert_count"):
            np.testing.assert_array_equal(v[name], got[0][0][name])
        np.testing.assert_array_equal(out, got[0][1])


@pytest.mark.parametrize("dt,S,H,I", [(2, 128, 64, 64), (2, 2048, 320, 448), (3, 1152, 192, 1216), (0, 640, 128, 320), (1, 2304, 1088, 1152)])
def test_dense_forward_leaves_the_routing_out(dt, S, H, I):
    """One expert in the dense packing: rows are tokens, nothing is routed. The bits of a routed forward, also between
    routed forwards (their counters), with the output laid over the input, and the same routing tables."""
    keys = _keys(S, H, I, 1, 1, act=1, dt=dt)
    c = moe_ref.cfg_from_keys(keys)
    x, wg, w_up, w_down, b_up, b_down = random_layer(c, seed=S + H, w_std=0.08, bias_std=0.1)
    iP = pack_inputs(c, x, wg * 0, w_up, w_down, b_up, b_down)
    dense = np.concatenate([iP[:S * H], iP[S * H + c.PX * H:]])
    d = ka.initialize(keys)
    try:
        oP, dev = synth.alloc_outputs(d), _to_device(c, iP)
        for _ in range(3):
            ka.moe.forward_host(dev, oP)
            ka.moe.stream_synchronize()
            want, views = _out_to_np(c, oP)[S * c.PX:].copy(), ka.moe.debug_views(d)
            buf = _to_device(c, dense)
            torch.cuda.synchronize()
            ka.moe.forward_host_dense(buf, buf[:S * H])
            ka.moe.stream_synchronize()
            np.testing.assert_array_equal(_out_to_np(c, buf)[:S * H], want)
            for name, value in ka.moe.debug_views(d).items():
                np.testing.assert_array_equal(value, views[name])
    finally:
        ka.finalize()


@pytest.mark.parametrize("mode", MODES, ids=MODE_IDS)
@pytest.mark.parametrize("dt", [0, 1], ids=["fp32", "tf32"])
@pytest.mark.parametrize("H,I,act", [(64, 128, 0), (192, 320, 1), (1024, 64, 1)])
def test_32_bit_tiles_of_few_rows(mode, dt, H, I, act):
    """32-row tiles whose K is shared out over four wavefronts: slices for two of them only, unequal numbers of
    slices, experts around the 32 rows they may hold."""
    _forced_rows(dt, H, I, [1, 31, 32, 33, 30, 32, 16, 17, 48, 40, 32, 32, 24, 56, 44, 44], cf=1.0, mode=mode, act=act)


@pytest.mark.parametrize("mode", MODES, ids=MODE_IDS)
@pytest.mark.parametrize("dt,H,I,rows,cf", [
    (2, 64, 4096, [96, 97, 127, 128, 64, 65, 100, 91], 1.5),                # 64 x 128 both ways: one column tile of 64 down
    (3, 320, 4160, [1, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 384], 2.0),   # 64 x 128 both ways, experts of up to six row blocks
    (2, 320, 6144, [1, 127, 128, 129, 255, 256, 257, 385, 512, 640], 2.5),  # 128 x 128 up, 64 x 128 down: row blocks of two smaller ones, the last of them cut short
    (2, 192, 4096, [2304], 1.0),                                           # one expert, its row blocks dealt to the queues, an odd last one
    (3, 192, 4096, [1792], 1.0),
], ids=lambda v: str(v) if not isinstance(v, list) else str(len(v)) + "e")
def test_down_projection_on_the_smaller_tile(mode, dt, H, I, rows, cf):
    """Wide up-projections whose long, few down-projection tiles leave CUs idle. (The other pairs with a smaller tile
    down: test_every_pair_of_16_bit_tiles_at_the_edges_of_its_rows.)"""
    _forced_rows(dt, H, I, rows, cf=cf, mode=mode)


@pytest.mark.parametrize("mode", MODES, ids=MODE_IDS)
@pytest.mark.parametrize("dt,S,H,I", [(2, 2304, 320, 448), (3, 1152, 1088, 192), (0, 640, 128, 320)])
def test_dense_output_over_its_inputs(mode, dt, S, H, I):
    """The dense packing with its output laid over other rows of x, over weights and biases, up to the last element of
    the inputs: every input is read before the output overwrites it, so the bits are those of an output
    of its own. (The output in place of x row for row: above.)"""
    keys = _keys(S, H, I, 1, 1, act=1, dt=dt)
    c = moe_ref.cfg_from_keys(keys)
    x, wg, w_up, w_down, b_up, b_down = random_layer(c, seed=S + I, w_std=0.08, bias_std=0.1)
    iP = pack_inputs(c, x, wg, w_up, w_down, b_up, b_down)
    dense = np.concatenate([iP[:S * H], iP[S * H + c.PX * H:]])
    per16 = 16 // dense.itemsize
    last = dense.size - S * H
    offsets = [per16, H, last // 2 // per16 * per16, last // per16 * per16]   # 16-byte aligned, as outputs have to be
    ka.initialize(keys)
    try:
        _apply(mode)
        own = torch.empty(S * H, dtype=_to_device(c, dense[:1]).dtype, device="cuda")
        ka.moe.forward_host_dense(_to_device(c, dense), own)
        ka.moe.stream_synchronize()
        want = _out_to_np(c, own)
        for at in offsets:
            buf = _to_device(c, dense)
            torch.cuda.synchronize()
            ka.moe.forward_host_dense(buf, buf[at:at + S * H])
            ka.moe.stream_synchronize()
            np.testing.assert_array_equal(_out_to_np(c, buf)[at:at + S * H], want, err_msg=f"output at element {at}")
    finally:
        ka.finalize()


@pytest.mark.parametrize("dt", [0, 2], ids=["fp32", "bf16"])
def test_dense_tokens_with_infinities_and_nan(dt):
    """Nothing is routed in the dense packing, in either mode: a token that holds an infinity or a NaN goes through both
    products like any other, and the other tokens keep their bits."""
    S, H, I = 640, 128, 192
    keys = _keys(S, H, I, 1, 1, act=0, dt=dt)
    tdt = {0: torch.float32, 2: torch.bfloat16}[dt]
    rng = np.random.default_rng(11)
    x, w_up, w_down = (torch.from_numpy(rng.standard_normal(n)).to(tdt) for n in ((S, H), (I, H), (H, I)))
    finite = x.clone()
    x[7, 3], x[300, 100], x[639, 0], x[64, 64] = float("inf"), -float("inf"), float("inf"), float("nan")
    special = [7, 64, 300, 639]
    h = x.double() @ w_up.double().T
    h = torch.where(h > 0, h, torch.zeros((), dtype=h.dtype))   # NaN gives 0, as in the kernels
    want = h @ w_down.double().T
    got = {}
    ka.initialize(keys)
    try:
        for name, values in (("finite", finite), ("special", x)):
            for mode, label in zip(MODES, MODE_IDS):
                _apply(mode)
                iP = torch.cat([values.flatten(), w_up.flatten(), w_down.flatten(), torch.zeros(H + I, dtype=tdt)]).cuda()
                oP = torch.empty(S * H, dtype=tdt, device="cuda")
                torch.cuda.synchronize()
                ka.moe.forward_host_dense(iP, oP)
                ka.moe.stream_synchronize()
                got[name, label] = oP.view(S, H).cpu()
    finally:
        ka.finalize()
    others = torch.ones(S, dtype=torch.bool)
    others[special] = False
    for label in MODE_IDS:
        out = got["special", label].double()
        for places in (torch.isnan, torch.isposinf, torch.isneginf):
            assert torch.equal(places(out), places(want)), label
        assert torch.equal(got["special", label][others], got["finite", label][others]), label


@pytest.mark.parametrize("where", ["x", "w_up", "one token"])
@pytest.mark.parametrize("exponent", [-124, -130, -135])
def test_tf32_operands_below_what_splits_exactly(where, exponent):
    """Operands whose remainder has bits below the last of a bf16 subnormal, against partners large enough for those bits
    to show: the products of the undivided operands, as on the fp32 matrix cores, with and without ordinary tokens beside."""
    S, H, I = 16384, 512, 512
    rng = np.random.default_rng(5)

    def values(*n):   # 11 significant bits, 1 <= |v| < 2
        return torch.from_numpy(rng.integers(1024, 2048, n) * rng.choice([-1.0, 1.0], n) / 1024)
    x, w_up, w_down = values(S, H), values(I, H), values(H, I) / 16
    small, large = 2.0 ** exponent, 2.0 ** 90
    if where == "x":
        x, w_up = x * small, w_up * large
    elif where == "w_up":
        x, w_up = x * large, w_up * small
    else:
        x[1000], w_up = x[1000] * small, w_up * large
        x[1001:] = x[1001:] / large
    x, w_up, w_down = x.float(), w_up.float(), w_down.float()
    iP = torch.cat([x.flatten(), w_up.flatten(), w_down.flatten(), torch.zeros(H + I)]).cuda()
    ka.initialize(_keys(S, H, I, 1, 1, act=0, dt=1))
    try:
        oP = torch.zeros(S * H, device="cuda")
        ka.moe.forward_host_dense(iP, oP)
        ka.moe.stream_synchronize()
        got = oP.view(S, H).cpu().double()
    finally:
        ka.finalize()

    def operand(v):
        return (v.view(torch.int32) & ~0x1fff).view(torch.float32).double()
    want = torch.relu(operand(x) @ operand(w_up).T) @ w_down.double().T
    rows = slice(None) if where != "one token" else slice(1000, 1001)
    # h is rounded to 11 bits on the way, 2^-11 of each of its values at most, and the output once more
    for part in (rows, slice(0, 1000), slice(1001, None)):
        assert float((got - want)[part].norm()) <= (2.0 ** -11 + 1e-5) * float(want[part].norm())


@pytest.mark.parametrize("operand", ["x", "w_up"])
@pytest.mark.parametrize("rows", ["of any scale", "growing", "starting with zeros", "shrinking", "of small values that show", "out of range"])
def test_tf32_rows_that_fit_fp16_and_rows_that_do_not(rows, operand):
    """The 256 x 256 tf32 tile scales every row by its first 32 values and multiplies in fp16. Rows of any scale fit; values far
    larger than the first ones, or so small beside them that fp16 cuts them, on their own or where the partners of the large ones
    are zero, and rows beyond 2^40 have to give what undivided products give, each row (column) to its own scale."""
    S, H, I = 16384, 512, 512
    rng = np.random.default_rng(13)

    def values(*n):   # 11 significant bits, 1 <= |v| < 2
        return torch.from_numpy(rng.integers(1024, 2048, n) * rng.choice([-1.0, 1.0], n) / 1024)
    x, w_up, w_down = values(S, H), values(I, H), values(H, I) / 16
    a, b = (x, w_up) if operand == "x" else (w_up, x)
    n = a.shape[0]
    some = torch.from_numpy(rng.choice(n, n // 3, replace=False))
    if rows == "of any scale":
        a *= 2.0 ** torch.from_numpy(rng.integers(-30, 31, (n, 1))).double()
    elif rows == "growing":
        a[some, 100:] *= 2.0 ** 12
    elif rows == "starting with zeros":
        a[some, :300] = 0.0
        a[some[:100]] = 0.0
    elif rows == "shrinking":
        a[some, 40:] *= 2.0 ** -30
    elif rows == "of small values that show":
        a[some, 40:] *= 2.0 ** -30
        b[:, :40] = 0.0
    else:
        a[some] *= 2.0 ** 50
    h = torch.relu(x @ w_up.T)
    scale = h.norm(dim=0)
    if operand == "w_up":   # every column of h counts as much as the others, whatever its scale
        w_down *= torch.where(scale > 0, 2.0 ** -torch.floor(torch.log2(scale.clamp_min(1e-300))), torch.ones(()).double())
    want = h @ w_down.T
    iP = torch.cat([x.flatten(), w_up.flatten(), w_down.flatten(), torch.zeros(H + I).double()]).float().cuda()
    keys = _keys(S, H, I, 1, 1, act=0, dt=1)
    _assert_tiles(keys, (3, 0))
    ka.initialize(keys)
    try:
        oP = torch.zeros(S * H, device="cuda")
        ka.moe.forward_host_dense(iP, oP)
        ka.moe.stream_synchronize()
        got = oP.view(S, H).cpu().double()
    finally:
        ka.finalize()
    ok = want.norm(dim=1) > 0
    assert torch.equal(got[~ok], want[~ok])
    # h is rounded to 11 bits on the way, 2^-11 of each of its values at most, and the output once more
    assert float(((got - want).norm(dim=1)[ok] / want.norm(dim=1)[ok]).max()) <= 2 * 2.0 ** -11


@pytest.mark.parametrize("small,base,p", [
    ("x", 0, 14), ("x", 0, 24), ("x", 0, 26), ("w_up", 0, 26), ("x", 0, 34), ("w_up", 0, 34),
    ("x", 0, 50), ("w_up", 0, 70),        # below what a second fp16 value holds
    ("x", 39, 150), ("w_up", 39, 158),    # nothing is left of them once their row is scaled
    ("x and w_up", 0, 18), ("x and w_up", 0, 30), ("x and w_up", 10, 60),
], ids=lambda v: str(v))
def test_tf32_sums_of_small_values_beside_large_sums(small, base, p):
    """Values from column 40 on 2^-p times the others, where every second row of the other operand is zero in front of column
    40: sums of the small values alone beside ordinary ones, in the same rows (columns). Each sum against its own products: a
    place of 11 bits for the rounding of h, 2^-19 of the products' magnitudes for 16 slices summed in fp32. w_down is the
    identity, which has h itself read back."""
    S, H, I = 16384, 512, 512
    rng = np.random.default_rng(17)

    def values(*n):   # 11 significant bits, 1 <= |v| < 2
        return torch.from_numpy(rng.integers(1024, 2048, n) * rng.choice([-1.0, 1.0], n) / 1024)
    x, w_up = values(S, H), values(I, H)
    for name, a, b in (("x", x, w_up), ("w_up", w_up, x)):
        if name in small.split(" and "):
            a *= 2.0 ** base
            a[:, 40:] *= 2.0 ** -p
            b[1::2, :40] = 0.0
    want, magnitude = torch.relu(x @ w_up.T), x.abs() @ w_up.T.abs()
    iP = torch.cat([x.flatten(), w_up.flatten(), torch.eye(H, dtype=torch.double).flatten(), torch.zeros(H + I).double()]).float().cuda()
    keys = _keys(S, H, I, 1, 1, act=0, dt=1)
    _assert_tiles(keys, (3, 0))
    ka.initialize(keys)
    try:
        oP = torch.zeros(S * H, device="cuda")
        ka.moe.forward_host_dense(iP, oP)
        ka.moe.stream_synchronize()
        got = oP.view(S, H).cpu().double()
    finally:
        ka.finalize()
    assert ((got - want).abs() <= 2.0 ** -11 * want + 2.0 ** -19 * magnitude).all()


@pytest.mark.parametrize("mode", MODES, ids=MODE_IDS)
@pytest.mark.parametrize("operand", ["x", "w_up"])
@pytest.mark.parametrize("rows", ["with a large channel", "starting with zeros", "starting with small values", "growing again and again"])
def test_tf32_rows_whose_first_values_do_not_stand_for_them(rows, operand, mode):
    """Rows that outgrow the scale of their first 32 values are scaled anew on the way: the rows (columns) beside them keep
    their bits, which another order of the sums would change, and every sum is within a place of 11 bits of h and 2^-19 of its
    products' magnitudes for 16 slices summed in fp32. w_down is the identity, which has h itself read back."""
    S, H, I = 16384, 512, 512
    rng = np.random.default_rng(19)
    x, w_up = torch.from_numpy(rng.standard_normal((S, H))), torch.from_numpy(rng.standard_normal((I, H)))

    def operands(x, w_up):   # 11 significant bits
        return [(v.float().view(torch.int32) & ~0x1fff).view(torch.float32).double() for v in (x, w_up)]
    plain = operands(x, w_up)
    a = x if operand == "x" else w_up
    some = torch.from_numpy(rng.choice(a.shape[0], a.shape[0] // 5, replace=False))
    if rows == "with a large channel":
        a[some, 300] *= 2.0 ** 12
    elif rows == "starting with zeros":
        a[some, :200] = 0.0
        a[some[::2], 200:] *= 8.0
    elif rows == "starting with small values":
        a[some, :32] *= 2.0 ** -12
    else:
        for at in (33, 100, 101, 479, 480):
            a[some, at:] *= 2.0 ** 7
    changed = operands(x, w_up)
    others = torch.ones(a.shape[0], dtype=torch.bool)
    others[some] = False
    keys = _keys(S, H, I, 1, 1, act=0, dt=1)
    _assert_tiles(keys, (3, 0))
    got = []
    ka.initialize(keys)
    try:
        _apply(mode)
        for xs, ws in (plain, changed):
            iP = torch.cat([xs.flatten(), ws.flatten(), torch.eye(H, dtype=torch.double).flatten(), torch.zeros(H + I).double()]).float().cuda()
            oP = torch.zeros(S * H, device="cuda")
            torch.cuda.synchronize()
            ka.moe.forward_host_dense(iP, oP)
            ka.moe.stream_synchronize()
            got.append(oP.view(S, H).cpu())
    finally:
        ka.finalize()
    same = (lambda h: h[others]) if operand == "x" else (lambda h: h[:, others])
    assert torch.equal(same(got[0]), same(got[1]))
    for (xs, ws), h in zip((plain, changed), got):
        want = torch.relu(xs @ ws.T)
        assert ((h.double() - want).abs() <= 2.0 ** -11 * want + 2.0 ** -19 * (xs.abs() @ ws.abs().T)).all()


@pytest.mark.parametrize("mode", MODES, ids=MODE_IDS)
@pytest.mark.parametrize("p", [46, 14, -14])
@pytest.mark.parametrize("S,H,I,E,act", [(16384, 320, 320, 64, 0), (4096, 1088, 1152, 16, 1)])
def test_tf32_tiles_that_are_scaled_anew_or_computed_again(mode, p, S, H, I, E, act):
    """Some hidden units 2^p as large, their weights down 2^-p: a layer whose output is of ordinary size, every second expert of which
    has rows of h (p > 0) or of w_down that outgrow their scale, and for p = 46 weights, and a growth of h, that fp16
    does not hold: both projections through the bf16 products. Routed tokens, slices that start at another K for
    every expert, row blocks and wavefronts cut short, biases."""
    edges = [1, 16, 17, 127, 128, 129, 130, 255, 256, 257, 300, 384, 385, 512]
    share, rest = divmod(S - sum(edges), E - len(edges))
    rows = edges + [share + 1] * rest + [share] * (E - len(edges) - rest)
    keys = _keys(S, H, I, E, 1, cf=2.0, act=act, dt=1)
    _assert_tiles(keys, (3, 0))
    c = moe_ref.cfg_from_keys(keys)
    iP = _one_hot_layer(c, rows, seed=37 + H)
    at = S * H + c.PX * H
    w_up, w_down = iP[at:at + E * I * H].reshape(E, I, H), iP[at + E * I * H:at + 2 * E * I * H].reshape(E, H, I)
    b_up = iP[at + 2 * E * I * H:at + 2 * E * I * H + E * I].reshape(E, I)
    units = [37, 100, 101, I - 3]
    w_up[::2, units] *= np.float32(2.0 ** p)
    b_up[::2, units] *= np.float32(2.0 ** p)
    w_down[::2, :, units] *= np.float32(2.0 ** -p)
    _, v, _, _ = check_against_oracle(c, keys, iP, mode)
    np.testing.assert_array_equal(v["expert_count"], np.array(rows))


@pytest.mark.parametrize("sign", [1, -1], ids=["positive", "negative"])
@pytest.mark.parametrize("low,high", [(0.001, 0.1), (0.1, 0.5), (0.5, 1.0), (1.0, 2.0)])
def test_gelu_keeps_the_bits_of_small_arguments(low, high, sign):
    """fp32, both projections the identity: no more than the roundings of 32-bit arithmetic between v Phi(v) and the
    result. Exponent (its last rounding only, of at most 2.7, times ln 2, below |v| = 1), exponential, product, difference
    and the fit's 2e-8: six of 2^-24 / sqrt 3 together in the mean square. Below -1 the difference of two numbers up to
    six times the result, and an exponent of up to 5.5, four times that; 0.5 v (1 + erff(v / sqrt 2)) has 2.7e-7 there."""
    S, H = 1024, 64
    v = torch.from_numpy(sign * np.random.default_rng(3).uniform(low, high, S * H)).float()
    eye = torch.eye(H)
    iP = torch.cat([v, eye.flatten(), eye.flatten(), torch.zeros(2 * H)]).cuda()
    ka.initialize(_keys(S, H, H, 1, 1, act=1, dt=0))
    try:
        oP = torch.empty(S * H, device="cuda")
        ka.moe.forward_host_dense(iP, oP)
        ka.moe.stream_synchronize()
        got = oP.cpu().double().numpy()
    finally:
        ka.finalize()
    v = v.double().numpy()
    want = v * 0.5 * erfc(-v / np.sqrt(2.0))
    rms = float(np.sqrt(np.mean(((got - want) / want) ** 2)))
    assert rms <= 6 ** 0.5 * 2.0 ** -24 / 3 ** 0.5 * (4 if low >= 1.0 and sign < 0 else 1), rms


@pytest.mark.parametrize("dt,S,H,E", [
    (2, 128, 64, 8), (2, 128, 448, 8), (3, 128, 832, 64),       # whole units whose shares are 0 to 4 steps
    (2, 8192, 1472, 16), (2, 8192, 1856, 40),                   # 5 and 6, 7 and 8 steps beside whole batches of 8 and of 4
    (3, 128, 3904, 16), (2, 128, 2944, 20), (3, 128, 1984, 8),  # spread tiles: 15 and 16, 11 and 12, 7 and 8 steps
    (0, 256, 320, 30), (1, 128, 704, 100),                      # 32-bit types: 16 values a step
], ids=lambda v: str(v))
def test_gate_shares_of_every_length(dt, S, H, E):
    """The steps of a share that do not fill a batch of loads, as runs of 8, 4, 2 and 1."""
    keys = _keys(S, H, 64, E, 1, dt=dt)
    c = moe_ref.cfg_from_keys(keys)
    iP = pack_inputs(c, *random_layer(c, seed=H + E, w_std=0.05, bias_std=0.1))
    check_against_oracle(c, keys, iP, ka.MODE_FUSED)


@pytest.mark.parametrize("schedule", [ka.SCHEDULE_DYNAMIC, ka.SCHEDULE_STATIC], ids=["dynamic", "static"])
@pytest.mark.parametrize("dt,S,H,I,E,k", [(2, 128, 1024, 2048, 16, 2), (3, 640, 448, 2816, 64, 2), (2, 2048, 1024, 4096, 1, 1), (0, 128, 256, 512, 8, 2)],
                         ids=lambda v: str(v))
def test_scheduler_statistics_count_tiles(dt, S, H, I, E, k, schedule):
    """kleos_scheduler_stats counts every tile once, whatever its size, also where the down-projection has one of its own."""
    keys = _keys(S, H, I, E, k, dt=dt)
    c = moe_ref.cfg_from_keys(keys)
    iP = _to_device(c, pack_inputs(c, *random_layer(c, seed=S + I, w_std=0.05)))
    d = ka.initialize(keys)
    try:
        ka.moe.set_schedule(schedule)
        ka.moe.forward_host_bench(iP, synth.alloc_outputs(d), skip=1, trials=2)
        st, v = ka.moe.scheduler_stats(), ka.moe.debug_views(d)
    finally:
        ka.finalize()
    kept = np.minimum(v["expert_count"].astype(np.int64), d.kept_capacity)
    tiles = ka.moe.debug_tiles(keys, torch.cuda.get_device_properties(0).multi_processor_count)
    (um, un), (dm, dn) = tiles["up"], tiles["down"]
    assert st["tiles"] == int((-(-kept // um)).sum()) * -(-I // un) + int((-(-kept // dm)).sum()) * -(-H // dn)


@pytest.mark.parametrize("schedule", [ka.SCHEDULE_DYNAMIC, ka.SCHEDULE_STATIC], ids=["dynamic", "static"])
@pytest.mark.parametrize("dt,S,H,I,E,k", [(2, 2304, 192, 4672, 16, 2), (3, 4608, 320, 2816, 16, 2), (2, 1664, 448, 1088, 40, 3), (0, 1152, 64, 576, 8, 2)], ids=lambda v: str(v))
def test_every_row_block_is_handed_out_once(dt, S, H, I, E, k, schedule):
    """Experts of two and more row blocks, which the static schedule takes in another order from round to round: as many tiles
    as there are, and the outputs of the launch-by-launch mode."""
    test_scheduler_statistics_count_tiles(dt, S, H, I, E, k, schedule)
    keys = _keys(S, H, I, E, k, dt=dt)
    c = moe_ref.cfg_from_keys(keys)
    iP = pack_inputs(c, *random_layer(c, seed=S + I, w_std=0.05, bias_std=0.1))
    outs = [check_against_oracle(c, keys, iP, mode)[2] for mode in ((ka.MODE_PHASED, ka.SCHEDULE_AUTO), (ka.MODE_FUSED, schedule))]
    np.testing.assert_array_equal(outs[0], outs[1])


@pytest.mark.parametrize("H,I,blocks,want", [
    (2368, 1536, [4] * 7 + [5], ka.SCHEDULE_DYNAMIC),   # 2 H + 3 I strided, 2 H + 2 I spread over the grid
    (1152, 2368, [4] * 7 + [5], ka.SCHEDULE_DYNAMIC),   # 3 H + 2 I : 2 H + 2 I, with an up-projection that sums less than half as long
    (2368, 256, [4] * 7 + [5], ka.SCHEDULE_STATIC),     # H + 3 I : H + 2 I, a round more that hardly counts
    (2368, 1536, [4] * 8, ka.SCHEDULE_STATIC),
], ids=lambda v: str(v))
def test_schedule_of_lists_that_end_unevenly(H, I, blocks, want):
    """Layers each of whose projections alone takes no queue longer than the grid (64 x 64 tiles, 64 workgroups to an XCD): what is
    strided and what is handed out goes by both together, in the values of K that a workgroup sums; outputs are those of the other mode."""
    assert torch.cuda.get_device_properties(0).multi_processor_count == 256
    last = 298 if blocks[-1] == 5 else 256
    rows = [(2048 - last) // 7] * 7 + [last]
    assert sum(rows) == 2048 and [-(-r // 64) for r in rows] == blocks
    keys = _keys(2048, H, I, 8, 1, cf=1.25, dt=0)
    assert ka.moe.debug_tiles(keys)["up"] == ka.moe.debug_tiles(keys)["down"] == (64, 64)
    c = moe_ref.cfg_from_keys(keys)
    iP = _to_device(c, _one_hot_layer(c, rows, seed=H))
    outs = []
    d = ka.initialize(keys)
    try:
        for mode in (ka.MODE_PHASED, ka.MODE_FUSED):
            ka.moe.set_mode(mode)
            oP = synth.alloc_outputs(d)
            ka.moe.forward_host(iP, oP)
            ka.moe.stream_synchronize()
            outs.append(_out_to_np(c, oP))
        assert ka.moe.schedule_taken() == want
    finally:
        ka.finalize()
    np.testing.assert_array_equal(outs[0], outs[1])


@pytest.mark.parametrize("mode", MODES, ids=MODE_IDS)
@pytest.mark.parametrize("E,counters", [(62, 496), (63, 504)])
def test_readiness_counters_on_either_side_of_their_lines(mode, E, counters):
    """Eight row blocks to an expert, as many counters as the scheduler's spare words hold and a few more: every tile is
    worked on once, launch after launch."""
    keys = _keys(4096, 64, 192, E, 1, cf=7.5, dt=0)
    c = moe_ref.cfg_from_keys(keys)
    assert ka.moe.debug_tiles(keys)["up"] == (64, 64) and E * -(-min(c.EC, c.cap_rows) // 64) == counters
    edges = [c.EC, 1, 0, 64, 65, 449, 448]
    share, rest = divmod(4096 - sum(edges), E - len(edges))
    rows = [share + 1] * rest + [share] * (E - len(edges) - rest) + edges
    _, v, _, _ = check_against_oracle(c, keys, _one_hot_layer(c, rows, seed=E), mode, launches=3)
    np.testing.assert_array_equal(v["expert_count"], np.array(rows))


def _assert_tiles(keys, want):
    t = ka.moe.debug_tiles(keys, torch.cuda.get_device_properties(0).multi_processor_count)
    tall = ("tall",) if t["variant"] == 4 and t["up"][0] == 256 else ()
    assert (t["variant"], t["down_small"], *tall) == want, f"the layer runs on {t}: another layer is needed for these tiles"


_ROWS_256 = [1, 15, 16, 17, 31, 33, 47, 48, 49, 63, 64, 65, 100, 127, 128, 129, 192, 193, 255, 256, 257]
_ROWS_128 = [1, 15, 16, 17, 31, 33, 47, 48, 49, 63, 64, 65, 79, 81, 100, 127, 128, 129]
_ROWS_64 = [1, 15, 16, 17, 31, 33, 47, 48, 49, 63, 64, 65]


@pytest.mark.parametrize("mode", MODES, ids=MODE_IDS)
@pytest.mark.parametrize("dt", [2, 3], ids=["bf16", "fp16"])
@pytest.mark.parametrize("want,S,H,I,E,cf,edges", [
    ((0, 0), 5120, 192, 448, 32, 3.0, _ROWS_256),       # 256 x 256, a last column tile of 192; experts of two row blocks
    ((0, 0), 5120, 448, 192, 32, 4.0, _ROWS_256),
    ((1, 0), 2048, 192, 704, 48, 4.0, _ROWS_128),       # 128 x 256
    ((1, 0), 1536, 704, 64, 64, 4.0, _ROWS_64),
    ((1, 1), 2048, 192, 2112, 48, 4.0, _ROWS_128),      # 128 x 256 up, 128 x 128 down
    ((2, 0), 5120, 192, 192, 8, 4.0, [1, 129, 257, 700, 1024, 1025]),
    ((2, 1), 5120, 192, 2048, 24, 3.0, _ROWS_256[-12:]),   # 256 x 256 up, 128 x 256 down
    ((4, 0), 1024, 192, 320, 16, 4.0, [1, 63, 64, 65, 111, 112, 113, 127, 128, 129]),   # 128 x 128
    ((4, 1), 2048, 192, 4160, 16, 4.0, [1, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 257]),   # 128 x 128 up, 64 x 128 down
    ((5, 0), 1024, 192, 320, 48, 4.0, _ROWS_64),        # 64 x 128
    ((6, 0), 128, 1088, 2112, 24, 6.0, [1, 15, 16, 17, 31, 33]),   # 64 x 128, weights non-temporal
    ((6, 0), 128, 1088, 2112, 24, 24.0, [63, 65]),
], ids=lambda v: v if isinstance(v, str) else (f"{v[0]}/{v[1]}" if isinstance(v, tuple) else str(len(v)) + "e" if isinstance(v, list) else str(v)))
def test_every_pair_of_16_bit_tiles_at_the_edges_of_its_rows(mode, dt, want, S, H, I, E, cf, edges):
    """Experts that end at and around the 16 rows of a matrix instruction, the 64 of a wavefront and the rows of a
    tile, on the tiles that each row names, which the choice of the library is held to."""
    keys = _keys(S, H, I, E, 1, cf=cf, act=1, dt=dt)
    _assert_tiles(keys, want)
    c = moe_ref.cfg_from_keys(keys)
    share, rest = divmod(S - sum(edges), E - len(edges))
    rows = edges + [share + 1] * rest + [share] * (E - len(edges) - rest)
    assert max(rows) <= c.EC
    _, v, _, _ = check_against_oracle(c, keys, _one_hot_layer(c, rows, seed=S + H), mode)
    np.testing.assert_array_equal(v["expert_count"], np.array(rows))


@pytest.mark.parametrize("mode", MODES, ids=MODE_IDS)
@pytest.mark.parametrize("dt", [2, 3], ids=["bf16", "fp16"])
@pytest.mark.parametrize("S,H,I,cf,down,edges", [
    (5120, 192, 704, 2.0, (256, 128), _ROWS_256[:12]),
    (5120, 192, 704, 2.0, (256, 128), _ROWS_256[-12:]),
    (5632, 704, 64, 2.4, (256, 128), _ROWS_256[-12:]),      # half a column tile and one slice of K
    (5632, 64, 1344, 2.0, (256, 128), _ROWS_256[-12:]),
    (5120, 192, 4160, 2.0, (64, 128), _ROWS_256[-12:]),     # the down-projection in quarters of a row block
], ids=lambda v: str(len(v)) + "e" if isinstance(v, list) else str(v))
def test_tall_tiles_at_the_edges_of_their_rows(mode, dt, S, H, I, cf, down, edges):
    """256 x 128 tiles, at the edges of the 16 rows of a matrix instruction, the 64 of a wavefront and the tile."""
    E = 24
    keys = _keys(S, H, I, E, 1, cf=cf, act=1, dt=dt)
    t = ka.moe.debug_tiles(keys, torch.cuda.get_device_properties(0).multi_processor_count)
    assert (t["variant"], t["up"], t["down"]) == (4, (256, 128), down)
    c = moe_ref.cfg_from_keys(keys)
    share, rest = divmod(S - sum(edges), E - len(edges))
    rows = edges + [share + 1] * rest + [share] * (E - len(edges) - rest)
    assert max(rows) <= c.EC
    _, v, _, _ = check_against_oracle(c, keys, _one_hot_layer(c, rows, seed=S + H), mode)
    np.testing.assert_array_equal(v["expert_count"], np.array(rows))


@pytest.mark.parametrize("mode", MODES, ids=MODE_IDS)
@pytest.mark.parametrize("dt", [2, 3], ids=["bf16", "fp16"])
@pytest.mark.parametrize("projection", ["up", "down"])
@pytest.mark.parametrize("K", [128, 192, 256])
def test_tall_tiles_sum_short_k_in_halves(mode, dt, projection, K):
    """Tall tiles form the sums of the two halves of K apart, as the 128-row tiles in whose place they run, also where K is two
    or three slices: 2^15 in the first slice, and 2^-9 in both matrix instructions of the last. In one run of fp32 sums each of
    the small products is lost, half of the last place of 2^15 that they are; in halves their sum arrives. All values are exact."""
    S, N = 6144, 1216
    H, I = (K, N) if projection == "up" else (N, K)
    keys = _keys(S, H, I, 1, 1, act=0, dt=dt)
    t = ka.moe.debug_tiles(keys, torch.cuda.get_device_properties(0).multi_processor_count)
    assert (t["variant"], t["up"], t["down"]) == (4, (256, 128), (256, 128))
    c = moe_ref.cfg_from_keys(keys)
    factors, w = np.zeros(K, np.float32), np.zeros((N, K), np.float32)
    factors[0], factors[[K - 64, K - 32]] = 256.0, 2.0 ** -5
    w[:, 0], w[:, [K - 64, K - 32]] = 128.0, 2.0 ** -4
    x, w_up, w_down, b_up, b_down = (np.zeros(n, np.float32) for n in ((S, H), (I, H), (H, I), I, H))
    if projection == "up":
        x[:], w_up, b_up[:], w_down[:, 5] = factors, w, -2.0 ** 15, 1.0
    else:
        b_up, w_down, b_down[:] = factors, w, -2.0 ** 15
    _, oP, _ = run_gpu(keys, _to_device(c, pack_inputs(c, x, np.zeros((1, H), np.float32), w_up, w_down, b_up, b_down)), mode)
    out = moe_ref.elems_to_f32(_out_to_np(c, oP), c)[S * c.PX:]
    np.testing.assert_array_equal(out, np.full(S * H, 2.0 ** -8, np.float32))


@pytest.mark.parametrize("mode", MODES, ids=MODE_IDS)
@pytest.mark.parametrize("dt", [2, 3], ids=["bf16", "fp16"])
@pytest.mark.parametrize("H,I", [(64, 128), (128, 64), (192, 320), (256, 64)])
def test_large_tiles_of_few_slices(mode, dt, H, I):
    """256 x 256 tiles whose loads end while the first slices are multiplied: one to five slices of K, with experts that
    end inside the upper and the lower half of a wavefront's rows and between them."""
    rows = [17, 193, 241, 256, 433, 700, 1025, 2255]
    keys = _keys(sum(rows), H, I, len(rows), 1, cf=4.0, act=0, dt=dt)
    _assert_tiles(keys, (2, 0))
    c = moe_ref.cfg_from_keys(keys)
    _, v, _, _ = check_against_oracle(c, keys, _one_hot_layer(c, rows, seed=H + I), mode)
    np.testing.assert_array_equal(v["expert_count"], np.array(rows))


@pytest.mark.parametrize("dt", [2, 3], ids=["bf16", "fp16"])
@pytest.mark.parametrize("want,S,H,I", [((2, 0), 6272, 704, 704), ((2, 1), 4224, 1088, 1216), ((4, 0), 3072, 64, 704), ((4, 1), 896, 320, 2432),
                                        ((4, 0, "tall"), 2176, 192, 1344), ((4, 1, "tall"), 1152, 64, 8192), ((4, 1, "tall"), 2176, 192, 4160),
                                        ((5, 0), 640, 320, 192)],
                         ids=lambda v: v if isinstance(v, str) else ("/".join(map(str, v)) if isinstance(v, tuple) else str(v)))
def test_dense_output_on_every_pair_of_tiles(dt, want, S, H, I):
    """The dense output is stored with a pitch of H where the routed forward stores pieces one tile wide: the bits of a
    routed forward on every pair of tiles that a single expert gets, with last row blocks and column tiles cut short."""
    keys = _keys(S, H, I, 1, 1, act=1, dt=dt)
    _assert_tiles(keys, want)
    c = moe_ref.cfg_from_keys(keys)
    x, wg, w_up, w_down, b_up, b_down = random_layer(c, seed=S + H, w_std=0.05, bias_std=0.1)
    iP = pack_inputs(c, x, wg * 0, w_up, w_down, b_up, b_down)
    dense = np.concatenate([iP[:S * H], iP[S * H + c.PX * H:]])
    d = ka.initialize(keys)
    try:
        for schedule in (ka.SCHEDULE_DYNAMIC, ka.SCHEDULE_STATIC):
            ka.moe.set_schedule(schedule)
            oP = synth.alloc_outputs(d)
            ka.moe.forward_host(_to_device(c, iP), oP)
            ka.moe.stream_synchronize()
            out = torch.empty(S * H, dtype=oP.dtype, device="cuda").fill_(float("nan"))
            torch.cuda.synchronize()
            ka.moe.forward_host_dense(_to_device(c, dense), out)
            ka.moe.stream_synchronize()
            np.testing.assert_array_equal(_out_to_np(c, out), _out_to_np(c, oP)[S * c.PX:])
    finally:
        ka.finalize()


@pytest.mark.parametrize("mode", MODES, ids=MODE_IDS)
@pytest.mark.parametrize("E", [96, 200, 320])
def test_tf32_large_tiles_with_many_experts(mode, E):
    """256 x 256 tiles on the 16-bit matrix cores with more than 64 experts: their workgroups of eight wavefronts hold two
    gate units of four at a time, in each of the three gates above 64 experts."""
    S, H, I = 16384, 128, 320
    keys = _keys(S, H, I, E, 4, cf=2.0, dt=1)
    _assert_tiles(keys, (3, 0))
    c = moe_ref.cfg_from_keys(keys)
    iP = pack_inputs(c, *random_layer(c, seed=E, w_std=0.08, bias_std=0.1))
    mask = np.zeros(c.S, np.uint8)
    mask[np.random.default_rng(E).choice(c.S, 600, replace=False)] = 1
    check_against_oracle(c, keys, iP, mode, token_mask=mask)


@pytest.mark.parametrize("mode", MODES, ids=MODE_IDS)
@pytest.mark.parametrize("E,H,cf", [(64, 64, 24.0), (300, 320, 96.0)])
def test_queues_with_experts_without_rows(mode, E, H, cf):
    """A workgroup looks for the segment of its next ticket from that of its last: queues whose experts hold no row in front
    of, between and behind those that do, and whole queues of them, whose workgroups take tiles of the others."""
    rows = [0] * E
    for e, n in ((0, 300), (8, 1), (24, 257), (40, 129), (E - 3, 128), (3, 64), (E - 1, 401)):
        rows[e] = n
    assert sum(rows) % 128 == 0
    _forced_rows(2, H, 576, rows, cf=cf, mode=mode)
