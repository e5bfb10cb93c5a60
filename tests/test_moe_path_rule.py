"""Which kernels the MoE layer and its two nodes take (no GPU needed: host arithmetic, for 256 compute units before a device is opened)."""
import random

import pytest

from tests._parity import moe_path

Q4, Q5, Q6, Q80 = 12, 13, 14, 8


# (type, experts, top_k, hidden, inter, tokens): us of the gate/up node on the decode launches | on the expert-grouped GEMM
@pytest.mark.parametrize("block", [(Q5, 16, 4, 3072, 256, 18),   # 17.9 | 27.1
                                   (Q5, 32, 2, 2048, 256, 46),   # 16.7 | 21.9
                                   (Q5, 8, 4, 3072, 512, 17),    # 21.0 | 26.6
                                   (Q6, 32, 2, 3072, 256, 47),   # 21.5 | 28.8
                                   (Q6, 32, 8, 2048, 256, 21),   # 19.1 | 24.2
                                   (Q5, 16, 2, 2048, 512, 35)])  # 18.6 | 23.0
def test_a_gateup_node_that_loses_on_the_gemm_stays_off_it(block):
    """Whatever stack follows it: a Q8_0 one makes up for nothing."""
    t, experts, k, hidden, inter, n = block
    assert moe_path(t, Q80, experts, hidden, inter, n, k)["gateup"] == 0 == moe_path(t, t, experts, hidden, inter, n, k)["gateup"]


@pytest.mark.parametrize("block", [(Q6, 128, 2, 2560, 512, 380),  # 102.5 | 61.2
                                   (Q4, 256, 6, 1280, 256, 246),  # 48.3 | 30.4
                                   (Q4, 64, 6, 2048, 512, 64), (Q4, 16, 8, 2816, 768, 24), (Q4, 16, 8, 2816, 768, 17),
                                   (Q4, 8, 2, 1280, 768, 27)])    # 54 pairs: 0.65 of the time
def test_a_gateup_node_that_gains_takes_it(block):
    t, experts, k, hidden, inter, n = block
    assert moe_path(t, Q80, experts, hidden, inter, n, k)["gateup"] == 1


def test_the_layer_takes_what_its_nodes_take():
    rng = random.Random(5)
    seen = set()
    for _ in range(6000):
        experts, k = rng.choice((4, 8, 16, 60, 128, 256, 512)), rng.choice((1, 2, 4, 8))
        t, d, n = rng.choice((Q4, Q5, Q6)), rng.choice((Q4, Q5, Q6)), int(2 ** rng.uniform(0, 12))
        p = moe_path(t, d, experts, 256 * rng.randint(1, 16), 256 * rng.randint(1, 6), n, k)
        assert (p["layer gateup"], p["layer down"]) == (p["gateup"], p["down"])
        assert n < 192 or p["gateup"] == p["down"]
        assert n > 8 or not p["gateup"]
        seen.add((p["gateup"], p["down"]))
    assert len(seen) == 4


def test_a_q80_down_stack_keeps_the_layer_on_the_decode_launches_below_192_tokens():
    rng = random.Random(6)
    for _ in range(1000):
        experts, n = rng.choice((8, 32, 256)), rng.randint(1, 400)
        p = moe_path(Q4, Q80, experts, 2048, 512, n, 8)
        assert p["down"] == 0 == p["layer down"]
        assert p["layer gateup"] == (moe_path(Q4, Q4, experts, 2048, 512, n, 8)["gateup"] if n >= 192 else 0)


@pytest.mark.parametrize("block,gemm", [((8, 2, 2048, 1024, 33), 0),   # 1.09 of the decode launches' time
                                        ((16, 2, 1024, 512, 32), 0),   # 1.05
                                        ((8, 2, 1280, 512, 35), 0),    # 1.07
                                        ((32, 2, 3072, 256, 47), 1),   # 0.93
                                        ((16, 4, 2560, 256, 20), 1),   # 0.61
                                        ((8, 4, 2048, 256, 26), 1)])   # 0.66
def test_a_down_product_of_several_wavefronts_a_row_stays_off_the_gemm(block, gemm):
    experts, k, hidden, inter, n = block
    assert moe_path(Q4, Q4, experts, hidden, inter, n, k)["down"] == gemm
