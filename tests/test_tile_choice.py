"""Which tiles a layer's expert projections run on (kleos_debug_tiles, no GPU needed): layers at which the choice was
measured against all others, and what it may never do."""
import random

import pytest

import aristos_amd as ka


def tiles(S, H, I, E, k, dt=2, cf=1.0, drop=1):
    return ka.moe.debug_tiles(ka.KleosConfig(capacity_factor=cf, drop_tokens=drop, expert_top_k=k, hidden_act=0, hidden_size=H,
                                             intermediate_size=I, mini_batch=1, num_experts=E, sequence_len=S, torch_dtype=dt))


@pytest.mark.parametrize("layer,want", [
    # experts of up to 64 rows on tiles of 64, not of 128 (62.6 : 70.3, 67.9 : 78.4 us per forward)
    (dict(S=128, H=2688, I=1024, E=8, k=3), (5, 0)),
    (dict(S=256, H=832, I=5952, E=8, k=1, drop=0), (5, 0)),
    # nothing dropped: hot experts may hold several times the mean (144.5 : 159.1, 94.4 : 105.0, 168.9 : 192.5)
    (dict(S=4096, H=1024, I=2048, E=32, k=2, drop=0), (2, 0)),
    (dict(S=6144, H=384, I=768, E=128, k=2, drop=0), (2, 0)),
    (dict(S=768, H=960, I=2496, E=64, k=6, cf=1.25, drop=0), (0, 0)),
    # a decode step through few large experts, bound by their weights (341 : 374 : 389 on 6, 5 and 1)
    (dict(S=128, H=4096, I=14336, E=8, k=2, drop=0), (6, 0)),
    # one long down-projection (62 : 71), the large batches
    (dict(S=2048, H=1024, I=4096, E=1, k=1), (4, 1)),
    (dict(S=8192, H=2048, I=2048, E=64, k=2), (0, 0)),
    (dict(S=8192, H=4096, I=14336, E=8, k=2, cf=1.25), (2, 0)),
    (dict(S=4096, H=7168, I=2048, E=256, k=8), (1, 0)),
], ids=str)
def test_measured_choices(layer, want):
    t = tiles(**layer)
    assert (t["variant"], t["down_small"]) == want


@pytest.mark.parametrize("layer,up,down", [
    # us per forward on 256 x 128 and on 128 x 128 tiles (with the down-projection on 64 x 128 ones, if it is, in both), weights from HBM
    (dict(S=2048, H=1024, I=4096, E=1, k=1), (256, 128), (64, 128)),     # 70.3 : 76.2
    (dict(S=1664, H=576, I=5120, E=1, k=1), (256, 128), (64, 128)),      # 70.5 : 73.6
    (dict(S=1408, H=832, I=1152, E=16, k=2), (256, 128), (256, 128)),    # 55.6 : 59.0
    (dict(S=1024, H=2624, I=6592, E=1, k=1, drop=0), (128, 128), (128, 128)),    # 162 : 147
    # strided through on one of the two only, handed out on the other
    (dict(S=2304, H=384, I=384, E=4, k=4), (256, 128), (256, 128)),      # 48.3 : 68.5
    (dict(S=1152, H=640, I=2752, E=1, k=1, cf=1.25), (256, 128), (64, 128)),     # 49.7 : 64.3
    (dict(S=3072, H=2240, I=832, E=1, k=1, cf=1.25), (128, 128), (128, 128)),    # 93.3 : 73.3
    (dict(S=1024, H=576, I=7552, E=1, k=1, cf=2.0), (128, 128), (64, 128)),      # 91.6 : 76.5
    (dict(S=128, H=512, I=9728, E=8, k=8), (128, 128), (64, 128)),       # 158 : 154, experts of one low row block
], ids=str)
def test_tall_tiles_where_they_save_rounds(layer, up, down):
    t = tiles(**layer)
    assert (t["variant"], t["up"], t["down"]) == (4, up, down)


def test_every_layer_gets_tiles_its_type_has():
    rng = random.Random(1)
    for _ in range(2000):
        E = rng.choice((1, 2, 8, 16, 64, 200, 512))
        layer = dict(S=128 * rng.randint(1, 64), H=64 * rng.randint(1, 64), I=64 * rng.randint(1, 128), E=E,
                     k=rng.randint(1, min(E, 8)), dt=rng.randint(0, 3), cf=rng.choice((1.0, 1.25, 2.0)), drop=rng.randint(0, 1))
        t = tiles(**layer)
        assert t["variant"] in {0: (0, 7), 1: (0, 3, 7), 2: (0, 1, 2, 4, 5, 6), 3: (0, 1, 2, 4, 5, 6)}[layer["dt"]], layer
        assert t["down_small"] == 0 or t["variant"] in (1, 2, 4), layer
        assert (t["up"] == t["down"]) == (t["down_small"] == 0), layer


def test_bad_arguments_are_refused():
    with pytest.raises(ka.KleosError):
        tiles(S=128, H=64, I=64, E=4, k=8)
    with pytest.raises(ka.KleosError):
        ka.moe.debug_tiles(ka.KleosConfig(sequence_len=128, hidden_size=64, intermediate_size=64, num_experts=4), compute_units=0)
