"""Prefill work items and gate/up forms at the sizes where the rule changes (needs an MI355X).

Items hold up to 32 pairs in calls of fewer than 224 tokens over at most 112 experts and
up to 64 in others; small items read their activations directly below 152 tokens and,
below 256, over more than 224 experts, and through LDS elsewhere.  Eight hot experts take
every token (items of 32 or 64 pairs and one remainder each), or the routing is flat (many
items of a few pairs), or a given number of experts shares the pairs but for one that takes
every token; the context is sized for exactly T tokens.
"""
import numpy as np
import pytest

import oracle as O
import qe_moe

pytestmark = pytest.mark.gpu
SEED = 0x17E35


def check_layer(torch, T, bias, used=None):
    L = O.SynthLayer(SEED, 0, bias=bias)
    m = qe_moe.MoE(n_layers=1, t_max=T)
    try:
        m.synth_layer(0, SEED, bias)
        x = O.gen_x(SEED, T, T)
        xd = torch.from_numpy(x).cuda()
        y = torch.empty_like(xd)
        for _ in range(2):  # the second call finds the counts of the first
            m.forward_normed(0, xd, y, T)
        torch.cuda.synchronize()
        g = m.routing(T)
        m.check()
    finally:
        m.close()
    o = O.moe_layer(L, x)
    assert used is None or np.unique(o["ids"]).size == used
    assert np.array_equal(g["ids"], o["ids"])
    assert np.array_equal(g["off"], o["off"]) and np.array_equal(g["pairs"], o["pairs"])
    # exact int8 block dots in both; fp32 sums in another order leave a few ulps, and an
    # h on a rounding step of its int8 scale now and then 1/127 of one element
    assert np.linalg.norm(y.cpu().numpy() - o["out"]) <= 1e-3 * np.linalg.norm(o["out"])


@pytest.mark.parametrize("hot", [True, False])
@pytest.mark.parametrize("T", [9, 16, 17, 31, 32, 97, 151, 152, 223, 224, 255, 256])
def test_items_at_rule_edges(torch_cuda, T, hot):
    print(f"items at T={T}, {'8 hot experts' if hot else 'flat routing'}", flush=True)
    bias = None
    if hot:
        bias = np.zeros(256, np.float32)
        bias[[0, 7, 63, 64, 130, 191, 192, 255]] = 50.0
    check_layer(torch_cuda, T, bias)


@pytest.mark.parametrize("T,used", [(96, 112), (96, 113), (151, 112), (152, 112), (152, 113), (223, 112), (223, 113),
                                    (224, 112), (223, 224), (223, 225), (255, 224), (255, 225), (256, 225)])
def test_items_by_experts_used(torch_cuda, T, used):
    print(f"items at T={T} over {used} experts", flush=True)
    bias = np.zeros(256, np.float32)
    pick = np.arange(used) * 256 // used
    bias[pick] = 50.0
    bias[pick[used // 2]] = 60.0
    check_layer(torch_cuda, T, bias, used)
