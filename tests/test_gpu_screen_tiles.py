"""The grouped screen at its edges, bit-exact to the oracle (needs an MI355X).

Two experts that every token routes to give tiles of exactly `tokens` pairs
(and a second tile past 16): the pair counts on both sides of the score
epilogue's one-item-per-lane rule (4 pairs for the point score, 12 for the
recovery-aware one). The hidden sizes give one block, an odd count below
eight, splits that end inside a two-block stage (span 3), splits without a
block, and the largest table; width 80 is five channel tiles, one past a
workgroup's four waves.
"""

import pytest

from calibration_free_moe.reader.budget import compile_budget
from tests.synthetic import make_layer
from tests.test_gpu_parity import assert_parity, build, run_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("score", ["point", "recovery-aware"])
@pytest.mark.parametrize("hidden,tokens", [
    (128, 4), (384, 13), (1152, 5), (2048, 4), (2048, 12), (2048, 17), (2176, 5), (2688, 13), (3072, 1),
    (3072, 3), (3072, 16), (3200, 1), (3968, 12),
])
def test_screen_tile_edges_bit_exact(hidden, tokens, score):
    # (the hidden sizes also cover the exact rows' part counts: 4 up to 2048, 6 up
    # to 3072, 8 above)
    layer = make_layer(hidden=hidden, width=80, experts=2, top_k=2, rank=16, tokens=tokens,
                       seed=300 + hidden + tokens)
    plan = compile_budget(hidden_size=hidden, expert_width=80, top_k=2, retention=0.25, screen_keep=0.625)
    reader = build(layer, plan, tokens, selection_score=score)
    out, expected = run_both(reader, layer, plan, layer.hidden, layer.ids, layer.weights)
    assert_parity(reader, out, expected, tokens)
